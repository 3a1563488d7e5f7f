"""Every kernel that the release build launches is launched by the build with host sanitizers too (no GPU: the host half of
each HIP file is compiled to assembly both ways, without inlining, and the launch stubs that it calls are compared).

clang's function sanitizer (part of -fsanitize=undefined) reads the words in front of an indirect callee; a kernel launched
through a function pointer has its handle there, a data object, and the optimiser drops the call without a word."""
import glob
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIP = os.path.join(ROOT, "alsparse_amd", "csrc", "hip")
HIPCC = os.path.join(os.environ.get("ROCM", "/opt/rocm"), "bin", "hipcc")


def _launched(path, *flags):
    r = subprocess.run([HIPCC, "--offload-arch=gfx950", "--cuda-host-only", "-O2", "-fno-inline", "-std=c++17", "-fPIC",
                        "-I" + os.path.join(ROOT, "include"), "-I/opt/rocm/include", "-Wno-unused-command-line-argument",
                        *flags, "-S", "-o", "-", path], stdout=subprocess.PIPE, stderr=subprocess.PIPE, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-3000:]
    return set(re.findall(r"(?:call|callq|jmp)\s+(\S*__device_stub__\S*?)(?:@PLT)?\s", r.stdout))


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="no HIP compiler")
@pytest.mark.parametrize("name", sorted(os.path.basename(f) for f in glob.glob(os.path.join(HIP, "*.hip"))))
def test_sanitized_host_code_launches_the_same_kernels(name):
    release = _launched(os.path.join(HIP, name))
    sanitized = _launched(os.path.join(HIP, name), "-Xarch_host", "-fsanitize=undefined")
    assert release, "no launch found in %s" % name
    assert sanitized == release, "launches that differ: %s" % sorted(sanitized ^ release)[:4]
