"""The fingerprint of a value array against the same sum in numpy: every word (or every word of the sample) counts once,
whatever the array's length and alignment -- last quads of one to three words, runs cut short, both kernels."""
import ctypes

import numpy as np
import pytest

from alsparse_amd import capi, hiprt
from helpers import announce

pytestmark = pytest.mark.gpu

GUARD_BYTES = 16384 + 64  # per-call scratch; the fingerprint lies behind 2 048 partial sums
FULL_BYTES = 32 << 20


def _fingerprint(words, run):
    n = words.size
    r = np.arange((n + run - 1) // run, dtype=np.uint64)
    slot = ((((r * np.uint64(2654435761)) & np.uint64(0xFFFFFFFF)) >> np.uint64(7)) & np.uint64(run // 64 - 1)) * np.uint64(64)
    pos = r * np.uint64(run) + slot
    pos = np.where(pos >= n, r * np.uint64(run), pos)
    idx = (pos[:, None] + np.arange(64, dtype=np.uint64)[None, :]).reshape(-1)
    idx = idx[idx < n]
    w = words[idx.astype(np.int64)]
    i = idx.astype(np.uint32)  # (positions below 2^32)
    t = i * np.uint32(0x85EBCA6B)
    a = (w ^ t) * np.uint32(0x9E3779B1)
    a ^= a >> np.uint32(15)
    b = (w + ((t >> np.uint32(7)) | (t << np.uint32(25)))) * np.uint32(0x27D4EB2F)
    b ^= b >> np.uint32(16)
    total = int((b.astype(np.uint64) << np.uint64(32) | a.astype(np.uint64)).sum(dtype=np.uint64))
    return total ^ (n * 0x9E3779B97F4A7C15 & (1 << 64) - 1)


@pytest.mark.parametrize("offset", [0, 1, 2, 4], ids=lambda o: "off%d" % o)
@pytest.mark.parametrize("words,full", [(1, 1), (2, 1), (3, 1), (4, 1), (5, 1), (63, 1), (66, 1), (255, 1), (1 << 20, 1),
                                        (2048 * 256 * 8 + 7, 1), (FULL_BYTES // 4 + 1, 0), (FULL_BYTES // 4 + 65, 0),
                                        (5 * (FULL_BYTES // 4) + 3, 0), (5 * (FULL_BYTES // 4) + 3, 1)])
def test_fingerprint_is_the_sum_over_the_words(gpu, words, full, offset):
    lib = capi.load()
    rng = np.random.default_rng(words + offset)
    host = rng.integers(0, 1 << 32, size=words + offset, dtype=np.uint32)
    nbytes = words * 4
    run = 64 if full or nbytes <= FULL_BYTES else int(lib.asamd_value_guard_run(nbytes)) // 4
    assert (run > 64) == (not full and nbytes >= FULL_BYTES + 256), "a sample"
    d, ws = hiprt.DeviceArray.from_numpy(host), hiprt.DeviceArray((GUARD_BYTES // 8,), np.uint64)
    stored = hiprt.DeviceArray.from_numpy(np.array([_fingerprint(host[offset:], run)], dtype=np.uint64))
    try:
        announce("fingerprint", words, "full", full, "offset", offset)
        at = ctypes.c_void_p(d.ptr + 4 * offset)
        assert lib.asamd_value_guard(None, at, nbytes, full, stored.c_ptr(), ws.c_ptr()) == 0
        got = ws.to_numpy()
        assert int(got[2048]) == int(stored.to_numpy()[0])
        assert got[2049:2050].view(np.int32)[0] == 0, "taken as changed"
    finally:
        for x in (d, ws, stored):
            x.free()


@pytest.mark.parametrize("dtype", [np.float32, np.complex128], ids=["f32", "c128"])
@pytest.mark.parametrize("flag", [None, 0, 1])
def test_a_flag_gates_the_gather(gpu, flag, dtype):
    """asamd_gather_values takes the address of a flag on the device, or nothing."""
    lib = capi.load()
    rng = np.random.default_rng(5)
    n, code = 70001, {"float32": 0, "complex128": 3}[np.dtype(dtype).name]
    host, perm = rng.integers(0, 1 << 20, size=n).astype(dtype), rng.permutation(n).astype(np.uint32)
    d = [hiprt.DeviceArray.from_numpy(v) for v in (host, perm, np.full(n, 7, dtype), np.array([flag or 0], np.int32))]
    try:
        announce("gather behind a flag", flag, np.dtype(dtype).name)
        assert lib.asamd_gather_values(None, code, 0, n, d[1].c_ptr(), d[0].c_ptr(), d[2].c_ptr(),
                                       None if flag is None else d[3].c_ptr()) == 0
        assert np.array_equal(d[2].to_numpy(), np.full(n, 7, dtype) if flag == 0 else host[perm])
    finally:
        for x in d:
            x.free()


@pytest.mark.parametrize("words", [5, 255, 70001, 2048 * 8 * 256 + 3])
def test_the_refreshing_kernel_works_out_the_verdict(gpu, words):
    """asamd_value_guard_begin leaves partial sums; the gather compares them with the recorded word in every workgroup, from one
    to as many as it launches, refreshes or does not, and leaves word and flag for the kernels behind and for the record."""
    lib = capi.load()
    rng = np.random.default_rng(words)
    host, perm = rng.standard_normal(words).astype(np.float32), rng.permutation(words).astype(np.uint32)
    want = _fingerprint(host.view(np.uint32), 64)
    d, dp = hiprt.DeviceArray.from_numpy(host), hiprt.DeviceArray.from_numpy(perm)
    ws, out, second = hiprt.DeviceArray((GUARD_BYTES // 8,), np.uint64), hiprt.DeviceArray((words,), np.float32), hiprt.DeviceArray((words,), np.float32)
    stored = hiprt.DeviceArray.from_numpy(np.zeros(1, np.uint64))
    old = np.full(words, 3, np.float32)
    try:
        for recorded, changed in ((want ^ 1, 1), (want, 0)):
            announce("verdict", words, changed)
            ws.copy_from(rng.integers(0, 1 << 63, GUARD_BYTES // 8).astype(np.uint64))
            stored.copy_from(np.array([recorded], np.uint64))
            out.copy_from(old)
            second.copy_from(old)
            check = capi.asamd_value_check()
            assert lib.asamd_value_guard_begin(None, d.c_ptr(), 4 * words, 0, stored.c_ptr(), ws.c_ptr(), ctypes.byref(check)) == 0
            assert check.words == words and check.settled == 0
            assert lib.asamd_gather_checked(None, 0, 0, words, dp.c_ptr(), d.c_ptr(), out.c_ptr(), ctypes.byref(check)) == 0
            check.settled = 1
            assert lib.asamd_gather_checked(None, 0, 0, words, dp.c_ptr(), d.c_ptr(), second.c_ptr(), ctypes.byref(check)) == 0
            hiprt.synchronize()
            assert int(stored.to_numpy()[0]) == recorded, "recorded before the copies are refreshed"
            assert lib.asamd_value_guard_commit(None, ws.c_ptr(), stored.c_ptr()) == 0
            hiprt.synchronize()
            for got in (out, second):
                assert np.array_equal(got.to_numpy(), host[perm] if changed else old)
            state = ws.to_numpy()
            assert int(state[2048]) == want and state[2049:2050].view(np.int32)[0] == changed
            assert int(stored.to_numpy()[0]) == want
    finally:
        for x in (d, dp, ws, out, second, stored):
            x.free()
