"""How the tiled layouts cut column blocks into chunks and hand them to the XCDs (tests/host_checks/tile_chunks.cpp, compiled
for the host and run: no GPU).  The reference has no counterpart."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host compiler")
def test_chunks_fill_rounds_and_are_handed_out_once(tmp_path):
    exe = str(tmp_path / "tile_chunks")
    r = subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-I" + os.path.join(ROOT, "alsparse_amd", "csrc", "hip"),
                        os.path.join(ROOT, "tests", "host_checks", "tile_chunks.cpp"), "-o", exe],
                       stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=120)
    assert r.returncode == 0, r.stdout[-3000:]
    r = subprocess.run([exe], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
