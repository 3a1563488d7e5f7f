"""Transposed CSR SpMV without an analysis where the sums are formed in LDS: the column slices (few entries; rows much
longer than the mean; few columns) at the edges of a chunk of 8 192 entries, of a slice and of the parts, and the
scatter's table in LDS (its slots meet, one or four rows per lane group, more entries than a table).  Against the oracle's
restatement of the reference's plain transposed kernel; sums are held in double precision, so the tolerance is the one of
every transposed product here."""
import ctypes
import time
from ctypes import byref, c_void_p

import numpy as np
import pytest

from alsparse_amd import capi, hiprt, workloads as wl
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


def rows_between_empty_ones(m, rows, lengths, cols, dt, base=0):
    """A matrix of m rows, all empty but the given ones."""
    per_row = np.zeros(m, np.int64)
    per_row[np.asarray(rows)] = lengths
    return csr_from_lengths(per_row.tolist(), cols, dt, base=base)


#: the rows that start over a chunk end at the walk's last row, one past it, far past it
EMPTY_ROWS = {
    "walked_to_the_end": lambda dt: rows_between_empty_ones(24577, [0, 24576], [200, 300], 400, dt),
    "one_more": lambda dt: rows_between_empty_ones(24578, [0, 24577], [200, 300], 400, dt),
    "last_walked_row_ends_the_chunk": lambda dt: rows_between_empty_ones(40000, [0, 24576, 24577, 39999], [8191, 1, 9000, 3], 9001, dt),
    "counted_and_walked": lambda dt: rows_between_empty_ones(42000, [0, 40959, 40960], [200, 300, 7], 400, dt),
    "one_more_than_walked": lambda dt: rows_between_empty_ones(42000, [0, 40960, 40961], [200, 300, 7], 400, dt),
    "empty_in_front": lambda dt: rows_between_empty_ones(300000, np.arange(290000, 300000), 4, 130, dt, base=1),
    "empty_behind": lambda dt: rows_between_empty_ones(300000, np.arange(10000), 4, 130, dt),
    "every_fortieth": lambda dt: rows_between_empty_ones(400000, np.arange(0, 400000, 40), 3, 300, dt),
    "runs": lambda dt: rows_between_empty_ones(200001, np.arange(200001)[(np.arange(200001) // 20000) % 2 == 1], 2, 3000, dt),
}


@pytest.mark.parametrize("entry", ["asamd_spmv_trans_slices", "asamd_spmv_trans_slices_gaps"], ids=["walked", "gaps"])
@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
@pytest.mark.parametrize("shape", sorted(EMPTY_ROWS))
def test_slices_over_long_runs_of_empty_rows(gpu, shape, dtype, entry):
    """Chunks over which more rows start than are walked look their entries' rows up."""
    a = EMPTY_ROWS[shape](dtype)
    code = capi.dtype_tag(a.dtype)
    x, y0 = wl.uniform(a.rows, dtype, 3), wl.uniform(a.cols, dtype, 4)
    da, lib, T = DeviceCsr(a), capi.load(), capi.scalar_type(dtype)
    dx, args = hiprt.DeviceArray.from_numpy(x), capi.asamd_spmv_args()
    part = hiprt.DeviceArray((max(1, lib.asamd_spmv_trans_slices_bytes(code, a.cols, a.nnz)),), np.uint8)
    try:
        for alpha, beta in ((1.0, 0.0), (2.0, 3.0)):
            announce("csrmv trans, empty rows", shape, np.dtype(dtype).name, alpha, beta)
            dy, al, be = hiprt.DeviceArray.from_numpy(y0), T(alpha), T(beta)
            args.dtype, args.m, args.n, args.nnz, args.base = code, a.rows, a.cols, a.nnz, a.base
            args.alpha, args.beta = ctypes.addressof(al), ctypes.addressof(be)
            args.val, args.row_ptr, args.col_ind, args.x, args.y = (v.ptr for v in (da.val, da.row_ptr, da.col, dx, dy))
            assert getattr(lib, entry)(None, byref(args), 0, part.c_ptr()) == 0
            hiprt.synchronize()
            check_trans(a, alpha, x, beta, y0, dy.to_numpy(), shape)
            dy.free()
    finally:
        part.free()
        dx.free()
        da.free()


def test_empty_rows_side_by_side_cost_no_more_than_the_scatter(gpu, monkeypatch):
    """4 M rows, all 400 000 entries in the last 100 000 of them and one long row, whose length makes the slices the choice:
    one part's workgroups met all the empty rows, and walked over them (40 times the scatter's time)."""
    a = rows_between_empty_ones(4000001, np.arange(3900001, 4000001), [4] * 99999 + [300], 15000, np.float32)
    assert capi.load().asamd_spmv_trans_slices_fit(0, a.rows, a.cols, a.nnz, 300) == 1
    x, y0 = wl.uniform(a.rows, a.dtype, 3), wl.uniform(a.cols, a.dtype, 4)
    best = []
    for switch in ("1", "0"):
        monkeypatch.setenv("ALSPARSE_AMD_XLDS", switch)  # 0: the scatter
        da = DeviceCsr(a)
        dx, dy = hiprt.DeviceArray.from_numpy(x), hiprt.DeviceArray.from_numpy(y0)
        al, be, descr = ctypes.c_float(1.0), ctypes.c_float(0.0), capi.make_descr()
        announce("empty rows side by side", switch)
        took = []
        for _ in range(6):
            hiprt.synchronize()
            t0 = time.perf_counter()
            for _ in range(10):
                assert capi.load().alphasparse_dcu_s_csrmv(gpu.h, T_, a.rows, a.cols, a.nnz, byref(al), byref(descr), da.val.c_ptr(),
                                                           da.row_ptr.c_ptr(), da.col.c_ptr(), None, dx.c_ptr(), byref(be),
                                                           dy.c_ptr()) == 0
            hiprt.synchronize()
            took.append(time.perf_counter() - t0)
        check_trans(a, 1.0, x, 0.0, y0, dy.to_numpy(), "switch " + switch)
        best.append(min(took[1:]))
        for d in (dx, dy):
            d.free()
        da.free()
    assert best[0] <= 2.0 * best[1], best
