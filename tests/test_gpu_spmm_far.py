"""Sparse times dense with B of 2 GiB and more (64-bit addresses instead of offsets into a buffer), and widths whose last chunk
of columns is narrower than one 128-bit load.  Few rows of B far apart, or few of many rows used, so that the host side stays
small; compared with the CPU oracle."""
import ctypes
from ctypes import byref

import numpy as np
import pytest

from alsparse_amd import capi, hiprt, workloads as wl
from helpers import DeviceCsr, announce
from oracle import oracle as orc

pytestmark = pytest.mark.gpu

DTYPES = {"f32": np.float32, "f64": np.float64, "c64": np.complex64, "c128": np.complex128}
ROW, COL = capi.ALPHA_SPARSE_LAYOUT_ROW_MAJOR, capi.ALPHA_SPARSE_LAYOUT_COLUMN_MAJOR


def _vector(n, dtype, stream):
    return wl.complex_vector(n, dtype, stream) if np.dtype(dtype).kind == "c" else wl.uniform(n, dtype, stream)


def _matrix(cols, dtype, base):
    """Rows around the blocks of sixteen entries and around the length from which a workgroup shares a row; columns may repeat."""
    rng = np.random.default_rng(3)
    lengths = np.array([0, 1, 15, 16, 17, 31, 40, 255, 256, 257, 0, 1025] + [20] * 57)
    row_ptr = np.concatenate([[0], np.cumsum(lengths)])
    col = rng.choice(cols, size=int(row_ptr[-1])).astype(np.int64)
    return row_ptr, col, _vector(col.size, dtype, 7), base


def _put(dev, at, host):
    host = np.ascontiguousarray(host)
    assert 0 <= at and at + host.nbytes <= dev.nbytes
    hiprt.check(hiprt.lib().hipMemcpy(ctypes.c_void_p(dev.ptr + at), host.ctypes.data_as(ctypes.c_void_p),
                                      ctypes.c_size_t(host.nbytes), ctypes.c_int(hiprt.H2D)), "hipMemcpy H2D")


def _csrmm(h, da, layout, trans_b, alpha, dB, ldb, beta, C0, ldc, n, k):
    a, T, descr = da.a, capi.scalar_type(da.a.dtype), capi.make_descr(base=da.a.base)
    dC = hiprt.DeviceArray.from_numpy(C0)
    al, be = T(alpha), T(beta)
    st = getattr(capi.load(), "alphasparse_dcu_%s_csrmm" % capi.prefix(a.dtype))(
        h.h, 0, trans_b, layout, a.rows, n, k, a.nnz, byref(al), byref(descr), da.val.c_ptr(), da.row_ptr.c_ptr(),
        da.col.c_ptr(), dB.c_ptr(), ldb, byref(be), dC.c_ptr(), ldc)
    assert st == 0, "csrmm status %d" % st
    hiprt.synchronize()
    out = dC.to_numpy()
    dC.free()
    return out


def _check(small, alpha, B, beta, C0, C, what):
    """small: the matrix over the rows of B that are used; tolerance per element as for SpMV"""
    tol = 1e-4 if np.dtype(small.dtype).name in ("float32", "complex64") else 1e-12
    C0 = np.zeros_like(C0) if beta == 0 else C0
    ref = orc.csrmm_plain(small, alpha, np.ascontiguousarray(B), beta, np.ascontiguousarray(C0))
    err = orc.csrmm_err(small, alpha, np.ascontiguousarray(B), beta, np.ascontiguousarray(C0), np.ascontiguousarray(C), ref)
    assert err.zero_den_mismatch == 0 and err.full <= tol, "%s: %r" % (what, err)


def _widths(size, whole_lines):
    """Every number of column lanes, one and several chunks, and a last chunk narrower than a load (V elements)."""
    v = 16 // size
    widths = [2 * v + 1, 4 * v, 4 * v + 1, 8 * v - 1, 8 * v + 1, 16 * v]
    if whole_lines:  # chunks of 256 bytes
        return widths + [16 * v + 1] + {4: [961, 963, 1025], 8: [481, 545], 16: []}[size]
    return widths + [16 * v + 1, 24 * v + 3, 32 * v, 32 * v + 1] + {4: [3969], 8: [1985], 16: []}[size]  # of 512


@pytest.mark.parametrize("far", [False, True], ids=["near", "2GiB"])
@pytest.mark.parametrize("whole_lines", [True, False], ids=["lines", "ragged"])
@pytest.mark.parametrize("name", list(DTYPES))
def test_rows_of_b_in_place(gpu, name, whole_lines, far):
    """Row-major B, and column-major B^T with column-major C: seventeen rows of B, next to one another or 128 MiB apart."""
    dtype, k = np.dtype(DTYPES[name]), 17
    row_ptr, col, val, base = _matrix(k, dtype, 1)
    a = wl.Csr(len(row_ptr) - 1, k, (row_ptr + base).astype(np.int32), (col + base).astype(np.int32), val, base, "far")
    widths = _widths(dtype.itemsize, whole_lines)
    most = max(widths)
    step = (1 << 27) // dtype.itemsize if far else 0  # sixteen steps of 128 MiB: 2 GiB from the first row to the last
    da = DeviceCsr(a)
    dB = hiprt.DeviceArray(((k - 1) * (step + most + 64) + most,), dtype)
    try:
        for n in widths:
            ldb = step + (n + 31) // 32 * 32 + (0 if whole_lines else 1)
            if far:
                assert ((k - 1) * ldb + n) * dtype.itemsize >= 1 << 31
            B = _vector(k * n, dtype, 5).reshape(k, n)
            for r in range(k):
                _put(dB, r * ldb * dtype.itemsize, B[r])
            for beta in (0.0, 0.5):
                announce("spmm, B in place:", name, "whole lines" if whole_lines else "ragged", "ldb", ldb, "n", n, "beta", beta)
                ldc = n + 3
                C0 = _vector(a.rows * ldc, dtype, 4).reshape(a.rows, ldc)
                Cin = np.where(np.arange(ldc) < n, np.nan, C0).astype(dtype) if beta == 0 else C0
                out = _csrmm(gpu, da, ROW, 0, 1.25, dB, ldb, beta, Cin, ldc, n, k)
                _check(a, 1.25, B, beta, C0[:, :n], out[:, :n], "row-major n=%d" % n)
                assert np.array_equal(out[:, n:], C0[:, n:]), "padding columns of C were touched"
                ldc = a.rows + 2
                C0 = _vector(n * ldc, dtype, 6).reshape(n, ldc)
                Cin = np.where(np.arange(ldc) < a.rows, np.nan, C0).astype(dtype) if beta == 0 else C0
                out = _csrmm(gpu, da, COL, 1, 1.25, dB, ldb, beta, Cin, ldc, n, k)
                _check(a, 1.25, B, beta, C0[:, :a.rows].T, out[:, :a.rows].T, "column-major n=%d" % n)
                assert np.array_equal(out[:, a.rows:], C0[:, a.rows:]), "padding rows of C were touched"
    finally:
        dB.free()
        da.free()


@pytest.mark.parametrize("name,n,k", [("f32", 130, (1 << 22) + 5), ("f32", 32, (1 << 24) + 5), ("f32", 16, (1 << 25) + 5),
                                      ("f64", 66, (1 << 22) + 5)])
def test_panels_of_two_gib(name, n, k):
    """Column-major B and C: panels of 256, 128 and 64 bytes a row that span 2 GiB together; the matrix uses the first and
    the last rows of B.  A handle of its own, so that its workspace goes with it."""
    dtype, used = np.dtype(DTYPES[name]), 40
    row_ptr, col, val, base = _matrix(2 * used, dtype, 0)
    m = len(row_ptr) - 1
    small = wl.Csr(m, 2 * used, row_ptr.astype(np.int32), col.astype(np.int32), val, 0, "used rows")
    a = wl.Csr(m, k, row_ptr.astype(np.int32), np.where(col < used, col, k - 2 * used + col).astype(np.int32), val, 0, "far panels")
    B = _vector(2 * used * n, dtype, 5).reshape(n, 2 * used)
    hiprt.set_device(0)
    h, da, dB = capi.Handle(), DeviceCsr(a), hiprt.DeviceArray((n * k,), dtype)
    try:
        for c in range(n):
            _put(dB, c * k * dtype.itemsize, B[c, :used])
            _put(dB, ((c + 1) * k - used) * dtype.itemsize, B[c, used:])
        for beta in (0.0, 0.5):
            announce("spmm, panels of 2 GiB:", name, "n", n, "k", k, "beta", beta)
            C0 = _vector(n * m, dtype, 6).reshape(n, m)
            Cin = np.full_like(C0, np.nan) if beta == 0 else C0
            out = _csrmm(h, da, COL, 0, 1.25, dB, k, beta, Cin, m, n, k)
            _check(small, 1.25, B.T, beta, C0.T, out.T, "panels n=%d" % n)
    finally:
        hiprt.synchronize()
        dB.free()
        da.free()
        h.close()
