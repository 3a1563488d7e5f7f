"""Every kernel that the release build launches is launched by the build with host sanitizers too (no GPU: the host half of
each HIP file is compiled to assembly both ways, without inlining, and the launch stubs that it calls are compared).

clang's function sanitizer (part of -fsanitize=undefined) reads the words in front of an indirect callee; a kernel launched
through a function pointer has its handle there, a data object, and the optimiser drops the call without a word."""
import glob
import os
import re
import struct
import subprocess

import pytest

from alsparse_amd import build

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


READELF = os.path.join(os.environ.get("ROCM", "/opt/rocm"), "llvm", "bin", "llvm-readelf")


def _kernels(tmp_path):
    """{symbol: its metadata} of every gfx950 kernel in the built library, one code object per HIP file."""
    data = open(build.LIB_PATH, "rb").read()
    magic, found = b"__CLANG_OFFLOAD_BUNDLE__", {}
    for at in (m.start() for m in re.finditer(magic, data)):
        count, = struct.unpack_from("<Q", data, at + len(magic))
        p = at + len(magic) + 8
        for _ in range(count):
            offset, size, length = struct.unpack_from("<QQQ", data, p)
            triple = data[p + 24:p + 24 + length]
            p += 24 + length
            if b"gfx950" not in triple or size == 0:
                continue
            obj = tmp_path / "object"
            obj.write_bytes(data[at + offset:at + offset + size])
            notes = subprocess.run([READELF, "--notes", str(obj)], stdout=subprocess.PIPE, text=True, timeout=120).stdout
            for block in re.split(r"\n  - (?=\.)", notes[notes.index("amdhsa.kernels:"):])[1:]:
                found[re.search(r"\.symbol:\s+'?(\S+?)\.kd", block).group(1)] = block
    return found


@pytest.mark.skipif(not os.path.exists(READELF), reason="no llvm-readelf")
def test_the_transposed_products_of_small_matrices_take_no_hidden_arguments(tmp_path):
    """A kernel that asks for its grid brings 256 bytes of hidden arguments, which the host writes on every launch; a pair of
    products of a few thousand entries is its launches."""
    kernels = {n: b for n, b in _kernels(tmp_path).items()
               if re.search(r"csrmv_trans_(scatter|slices)_kernel|trans_partials_sum_kernel|scale_vec_kernel", n)}
    assert sum("trans_scatter" in n for n in kernels) >= 40 and sum("trans_slices" in n for n in kernels) == 12
    asking = [n for n, block in kernels.items() if "hidden_" in block]
    assert not asking, asking[:4]
