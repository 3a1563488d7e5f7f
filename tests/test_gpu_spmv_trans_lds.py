"""Transposed CSR SpMV without an analysis where the sums are formed in LDS: the column slices (few entries; rows much
longer than the mean; few columns) at the edges of a chunk of 8 192 entries, of a slice and of the parts, and the
scatter's table in LDS (its slots meet, one or four rows per lane group, more entries than a table).  Against the oracle's
restatement of the reference's plain transposed kernel; sums are held in double precision, so the tolerance is the one of
every transposed product here."""
from ctypes import byref, c_void_p

import numpy as np
import pytest

from alsparse_amd import capi, workloads as wl
from helpers import DeviceCsr, announce
from helpers_shapes import csr_from_lengths
from test_gpu_complex import H_, T_, check, complexify, oracle_mv, real_dtype, run_csrmv
from test_gpu_spmv_trans import check_trans, run_csrmv_trans

pytestmark = pytest.mark.gpu


def skewed(rows, cols, most, dt, base=0):
    """Rows of 0 .. 5 entries and a few of up to `most` (well beyond 16 times the mean)."""
    lengths = np.arange(rows) % 6
    lengths[rows // 3], lengths[rows - 1] = most, most // 2
    return csr_from_lengths(lengths.tolist(), cols, dt, base=base)


#: name: (matrix, whether the slices take it)
SHAPES = {
    "one_chunk": (lambda dt: csr_from_lengths([4] * 2048, 3000, dt), 1),
    "one_chunk_and_one": (lambda dt: csr_from_lengths([4] * 2047 + [0, 5], 3000, dt), 0),
    "few_columns_two_chunks": (lambda dt: csr_from_lengths([0, 0] + [64] * 256 + [0], 70, dt), 1),
    "few_columns_two_chunks_and_one": (lambda dt: csr_from_lengths([64] * 256 + [1], 256, dt), 1),
    "one_row_over_chunks": (lambda dt: csr_from_lengths([9000, 7000] + [0] * 100, 9001, dt), 1),
    "slices_end_inside": (lambda dt: csr_from_lengths([3] * 1000, 64 * 256 + 1, dt), 1),
    "skewed": (lambda dt: skewed(30011, 40009, 20000, dt), 1),
    "skewed_base_one": (lambda dt: skewed(9001, 20011, 9000, dt, base=1), 1),
    "few_columns": (lambda dt: csr_from_lengths([13] * 20011, 199, dt), 1),
    "few_columns_one": (lambda dt: csr_from_lengths([1] * 30001, 1, dt), 1),
    "table_narrow": (lambda dt: wl.laplace2d(301, 203, dt), 0),
    "table_one_row": (lambda dt: csr_from_lengths([20] * 5003, 5000, dt), 0),
    "table_four_rows": (lambda dt: csr_from_lengths(([9, 0, 40, 9] * 20003), 50021, dt), 0),
    "table_overflows": (lambda dt: csr_from_lengths([300] * 600, 30011, dt), 0),
}


@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
@pytest.mark.parametrize("shape", sorted(SHAPES))
def test_transposed_sums_in_lds(gpu, shape, dtype):
    make, slices = SHAPES[shape]
    a = make(dtype)
    longest = int(np.diff(a.row_ptr).max())
    code = {np.float32: 0, np.float64: 1}[dtype]
    assert capi.load().asamd_spmv_trans_slices_fit(code, a.rows, a.cols, a.nnz, longest) == slices
    x, y0 = wl.uniform(a.rows, dtype, 3), wl.uniform(a.cols, dtype, 4)
    da = DeviceCsr(a)
    try:
        for alpha, beta in ((1.0, 0.0), (2.0, 3.0), (-0.75, 1.0)):
            announce("csrmv trans, sums in LDS", shape, np.dtype(dtype).name, alpha, beta)
            y = run_csrmv_trans(gpu, da, alpha, x, beta, y0)
            check_trans(a, alpha, x, beta, y0, y, shape)
    finally:
        da.free()


@pytest.mark.parametrize("op", [T_, H_], ids=["T", "H"])
@pytest.mark.parametrize("dtype", [np.complex64, np.complex128], ids=["c64", "c128"])
@pytest.mark.parametrize("shape", ["one_chunk_and_one", "skewed_base_one", "few_columns", "table_one_row", "table_four_rows"])
def test_transposed_sums_in_lds_complex(gpu, shape, dtype, op):
    a = complexify(SHAPES[shape][0](real_dtype(dtype)), dtype)
    x, y0 = wl.complex_vector(a.rows, dtype, 3), wl.complex_vector(a.cols, dtype, 4)
    da = DeviceCsr(a)
    try:
        for alpha, beta in ((1.0, 0.0), (0.75 - 0.5j, 0.25 + 1.5j)):
            announce("csrmv, sums in LDS", shape, np.dtype(dtype).name, op, alpha, beta)
            y = run_csrmv(gpu, da, op, alpha, x, beta, y0)
            metric, ref = oracle_mv(a, op, alpha, x, beta, y0)
            check(metric, alpha, x, beta, y0, y, ref, shape)
    finally:
        da.free()


def test_the_route_is_settled_with_the_plan(gpu, monkeypatch):
    """A transposed multiply works nothing out anew: the scratch that a plan asks for stays what it was, whatever the
    switches say later."""
    a = SHAPES["skewed"][0](np.float32)
    lib, da, plan = capi.load(), DeviceCsr(a), c_void_p()
    try:
        announce("route of the transposed product")
        assert lib.asamd_csr_plan_create_dtype(None, a.rows, a.cols, a.nnz, da.row_ptr.c_ptr(), da.col.c_ptr(), None, a.base,
                                               capi.dtype_tag(a.dtype), 0, byref(plan)) == 0
        needed = lib.asamd_csr_plan_workspace_bytes(plan)
        assert needed > lib.asamd_spmv_trans_slices_bytes(0, a.cols, a.nnz) > 0
        monkeypatch.setenv("ALSPARSE_AMD_XLDS", "0")
        assert lib.asamd_csr_plan_workspace_bytes(plan) == needed
    finally:
        lib.asamd_csr_plan_destroy(plan)
        da.free()
