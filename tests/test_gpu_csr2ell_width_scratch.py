"""csr2ell_width's scratch is its own: the handle's buffer, which a multiply on another stream of the handle may still be using,
is left alone, and calls of several threads do not meet."""
import ctypes
import threading
from ctypes import byref, c_int32

import numpy as np
import pytest

from alsparse_amd import capi, hiprt
from helpers import announce

pytestmark = pytest.mark.gpu


def _width(h, d_rp, rows):
    d, w = capi.make_descr(), c_int32(-1)
    assert capi.load().alphasparse_dcu_csr2ell_width(h.h, rows, byref(d), d_rp.c_ptr(), byref(d), byref(w)) == 0
    return w.value


def _buffer(h):
    """(address, bytes) of the handle's buffer: the word behind its size, which is made one that nothing else in the record is."""
    size = (5 << 20) + 4096
    assert capi.load().asamd_handle_reserve(h.h, size) == 0
    word = lambda i: ctypes.c_uint64.from_address(ctypes.cast(h.h, ctypes.c_void_p).value + 8 * i).value
    i = 0
    while word(i) != size:  # (in the record, before its end)
        i += 1
    return word(i + 1), size


def test_the_handles_buffer_is_left_alone():
    hiprt.set_device(0)
    h = capi.Handle()
    rows = 600 * 2048
    lengths = np.random.default_rng(1).integers(0, 9, size=rows)
    d_rp = hiprt.DeviceArray.from_numpy(np.concatenate([[0], np.cumsum(lengths)]).astype(np.int32))
    try:
        at, size = _buffer(h)
        want = np.full(size, 0xA5, dtype=np.uint8)
        copy = lambda dst, src, kind: hiprt.check(hiprt.lib().hipMemcpy(dst, src, ctypes.c_size_t(size), ctypes.c_int(kind)), "hipMemcpy")
        copy(ctypes.c_void_p(at), want.ctypes.data_as(ctypes.c_void_p), hiprt.H2D)
        announce("csr2ell_width beside the handle's buffer")
        assert _width(h, d_rp, rows) == 8
        got = np.zeros_like(want)
        copy(got.ctypes.data_as(ctypes.c_void_p), ctypes.c_void_p(at), hiprt.D2H)
        assert np.array_equal(got, want)
    finally:
        d_rp.free()
        h.close()


def test_widths_of_two_threads():
    hiprt.set_device(0)
    rows, wrong = 1 << 20, []
    sides = []
    for longest in (7, 4001):
        lengths = np.full(rows, 2)
        lengths[rows - 1] = longest
        rp = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int32)
        sides.append((capi.Handle(), hiprt.DeviceArray.from_numpy(rp), longest))

    def calls(h, d_rp, longest):
        hiprt.set_device(0)
        wrong.extend(w for w in (_width(h, d_rp, rows) for _ in range(200)) if w != longest)

    try:
        announce("csr2ell_width from two threads")
        threads = [threading.Thread(target=calls, args=side) for side in sides]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert not wrong
    finally:
        for h, d_rp, _ in sides:
            d_rp.free()
            h.close()
