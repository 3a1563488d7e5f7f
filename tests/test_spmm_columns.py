"""Which columns of B and C the lanes of the sixteen-lane SpMM groups take, for every width up to 36 chunks and both address
forms, and which rows of A their workgroups (tests/host_checks/group_columns.hip, compiled for the host and run: no GPU)."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = os.path.join(os.environ.get("ROCM", "/opt/rocm"), "bin", "hipcc")


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="no HIP compiler")
def test_lane_columns_stay_inside_the_row_and_cover_it_once(tmp_path):
    exe = str(tmp_path / "group_columns")
    r = subprocess.run([HIPCC, "--offload-arch=gfx950", "--cuda-host-only", "-O1", "-std=c++17", "-Wno-unused-command-line-argument",
                        "-I" + os.path.join(ROOT, "include"), "-I" + os.path.join(ROOT, "alsparse_amd", "csrc", "hip"),
                        os.path.join(ROOT, "tests", "host_checks", "group_columns.hip"), "-o", exe],
                       stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=300)
    assert r.returncode == 0, r.stdout[-3000:]
    r = subprocess.run([exe], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=120)
    assert r.returncode == 0, r.stdout
