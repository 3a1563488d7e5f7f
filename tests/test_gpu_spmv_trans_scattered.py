"""Transposed CSR SpMV without an analysis, chosen by the columns: slices with their sums in LDS where the columns are
scattered, the scatter with its table where neighbouring rows share them.  The sampled lines per entry against a count on
the host, the choice they lead to, and the public call against the oracle; sums are held in double precision, so the
tolerance is the one of every transposed product here."""
from ctypes import byref, c_float, c_int32

import numpy as np
import pytest

from alsparse_amd import capi, hiprt, workloads as wl
from helpers import DeviceCsr, announce
from helpers_shapes import csr_from_lengths
from test_gpu_complex import H_, T_, check, complexify, oracle_mv, real_dtype, run_csrmv
from test_gpu_spmv_trans import check_trans, run_csrmv_trans

pytestmark = pytest.mark.gpu

CODES = {np.float32: 0, np.float64: 1, np.complex64: 2, np.complex128: 3}
WORDS = 37  # row statistics and the lines

#: name: (matrix, whether the slices take it)
SHAPES = {
    "scattered": (lambda dt: csr_from_lengths([30] * 9001, 12007, dt), 1),
    "scattered_base_one": (lambda dt: csr_from_lengths([31] * 9001, 12007, dt, base=1), 1),
    "scattered_three_slices": (lambda dt: csr_from_lengths([25, 0, 40] * 9001, 50021, dt), 1),
    "short_rows_many_columns": (lambda dt: csr_from_lengths([3] * 30011, 150011, dt), 0),
    "fewer_than_the_runs": (lambda dt: csr_from_lengths([32] * 2047, 9001, dt), 0),
    "laplacian": (lambda dt: wl.laplace2d(301, 403, dt), 0),
}


def sampled_lines(a, dtype):
    """What 64 runs of 1 024 entries meet, counted on the host."""
    if a.nnz < 65536:
        return 0.0
    col = a.col_ind.astype(np.int64) - a.base
    begins = [(a.nnz - 1024) * b // 63 for b in range(64)]
    size = np.dtype(dtype).itemsize
    return sum(np.unique(col[b:b + 1024] * size // 128).size for b in begins) / 65536.0


def device_lines(da, a, dtype):
    lib = capi.load()
    scratch = hiprt.DeviceArray.from_numpy(np.zeros(WORDS, np.int32))
    stats, lines = (c_int32 * WORDS)(), c_float(-1.0)
    try:
        assert lib.asamd_csr_row_stats_lines(None, a.rows, da.row_ptr.ptr, a.nnz, a.base, np.dtype(dtype).itemsize,
                                             da.col.ptr, scratch.ptr, stats, byref(lines)) == 0
    finally:
        scratch.free()
    lengths = np.diff(a.row_ptr)
    assert (stats[0], stats[1], stats[2]) == (lengths.min(), lengths.max(), a.row_ptr[0])
    return lines.value


@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
@pytest.mark.parametrize("shape", sorted(SHAPES))
def test_transposed_by_columns(gpu, shape, dtype):
    make, slices = SHAPES[shape]
    a = make(dtype)
    x, y0 = wl.uniform(a.rows, dtype, 3), wl.uniform(a.cols, dtype, 4)
    da = DeviceCsr(a)
    try:
        lines, want = device_lines(da, a, dtype), sampled_lines(a, dtype)
        # fewer lines than the bitmap's 2^15 bits: no two share one
        assert abs(lines - want) < 1e-6
        assert capi.load().asamd_spmv_trans_slices_pay(CODES[dtype], a.cols, a.nnz, lines) == slices
        for alpha, beta in ((1.0, 0.0), (2.0, 3.0), (-0.75, 1.0)):
            announce("csrmv trans by columns", shape, np.dtype(dtype).name, alpha, beta)
            check_trans(a, alpha, x, beta, y0, run_csrmv_trans(gpu, da, alpha, x, beta, y0), shape)
    finally:
        da.free()


@pytest.mark.parametrize("op", [T_, H_], ids=["T", "H"])
@pytest.mark.parametrize("dtype", [np.complex64, np.complex128], ids=["c64", "c128"])
@pytest.mark.parametrize("shape", ["scattered_base_one", "scattered_three_slices", "laplacian"])
def test_transposed_by_columns_complex(gpu, shape, dtype, op):
    a = complexify(SHAPES[shape][0](real_dtype(dtype)), dtype)
    x, y0 = wl.complex_vector(a.rows, dtype, 3), wl.complex_vector(a.cols, dtype, 4)
    da = DeviceCsr(a)
    try:
        lines = device_lines(da, a, dtype)
        assert capi.load().asamd_spmv_trans_slices_pay(CODES[dtype], a.cols, a.nnz, lines) == SHAPES[shape][1]
        for alpha, beta in ((1.0, 0.0), (0.75 - 0.5j, 0.25 + 1.5j)):
            announce("csrmv by columns", shape, np.dtype(dtype).name, op, alpha, beta)
            y = run_csrmv(gpu, da, op, alpha, x, beta, y0)
            metric, ref = oracle_mv(a, op, alpha, x, beta, y0)
            check(metric, alpha, x, beta, y0, y, ref, shape)
    finally:
        da.free()
