"""Small analysed transposed products read the caller's values through the copy's permutation: by lane groups (one to eight
trips of four entries per lane, wider groups for longer rows) or, where a row of A^T would keep a wave longer, by the merge
path.  Any values with the analysed structure give their own product, without a second analysis; results are reproducible."""
from ctypes import byref, c_void_p

import numpy as np
import pytest

from alsparse_amd import capi, hiprt, workloads as wl
from helpers import DeviceCsr, announce
from helpers_shapes import csr_from_lengths
from oracle import oracle as orc
from test_gpu_complex import H_, T_, check, complexify, oracle_mv, real_dtype, run_csrmv
from test_gpu_spmv_trans import check_trans

pytestmark = pytest.mark.gpu


def transposed_lengths(lengths, rows, dt, base=0):
    """A matrix of `rows` rows whose transpose has rows of the given lengths."""
    at = csr_from_lengths(lengths, rows, dt)
    a = orc.transpose(at)
    return wl.Csr(a.rows, a.cols, (a.row_ptr + base).astype(np.int32), (a.col_ind + base).astype(np.int32), a.values, base,
                  "transposed " + at.name)


SHAPES = {
    "short_rows": lambda dt: transposed_lengths([0, 1, 2, 3, 4, 5, 0, 7] * 130, 900, dt),
    "base_one": lambda dt: transposed_lengths([3, 0, 6] * 211, 401, dt, base=1),
    "a_trip_and_one": lambda dt: transposed_lengths([8, 9, 31, 32, 33] * 41, 601, dt),
    "wider_groups": lambda dt: transposed_lengths([2] * 3001 + [127, 128, 129], 700, dt),
    "eight_trips": lambda dt: transposed_lengths([2] * 3001 + [2048], 4001, dt),
    "merge_path": lambda dt: transposed_lengths([2] * 3001 + [2049, 0, 5000, 1], 6001, dt),
    "one_column": lambda dt: transposed_lengths([5000], 5000, dt),
    "largest": lambda dt: wl.uniform_rows(1 << 16, 70001, 8, dt),
    "one_more": lambda dt: transposed_lengths([8] * (1 << 16) + [1], 70001, dt),
}


@pytest.mark.parametrize("op", [T_, H_], ids=["T", "H"])
@pytest.mark.parametrize("dtype", [np.float32, np.float64, np.complex64, np.complex128], ids=["f32", "f64", "c64", "c128"])
@pytest.mark.parametrize("shape", sorted(SHAPES))
def test_small_analysed_transposed_products(gpu, shape, dtype, op):
    is_complex = np.dtype(dtype).kind == "c"
    if op == H_ and not is_complex:
        pytest.skip("real types have no conjugate transpose")
    a = SHAPES[shape](real_dtype(dtype) if is_complex else dtype)
    a = complexify(a, dtype) if is_complex else a
    draw = wl.complex_vector if is_complex else wl.uniform
    x, y0 = draw(a.rows, dtype, 3), draw(a.cols, dtype, 4)
    lib = capi.load()
    da = DeviceCsr(a)
    info = capi.alphasparse_dcu_mat_info_t()
    assert lib.alphasparse_dcu_create_mat_info(byref(info)) == 0
    try:
        descr = capi.make_descr(base=a.base)
        assert getattr(lib, "alphasparse_dcu_%s_csrmv_analysis" % capi.prefix(a.dtype))(
            gpu.h, op, a.rows, a.cols, a.nnz, byref(descr), da.val.c_ptr(), da.row_ptr.c_ptr(), da.col.c_ptr(), info) == 0

        def product(matrix, alpha, beta, what):
            announce("csrmv permuted", shape, np.dtype(dtype).name, op, what)
            y = run_csrmv(gpu, da, op, alpha, x, beta, y0, info)
            if is_complex:
                metric, ref = oracle_mv(matrix, op, alpha, x, beta, y0)
                check(metric, alpha, x, beta, y0, y, ref, "%s %s" % (shape, what))
            else:
                check_trans(matrix, alpha, x, beta, y0, y, "%s %s" % (shape, what))
            return y

        product(a, 1.0, 0.0, "beta 0")
        first = product(a, 2.0, 3.0, "beta 3")
        assert np.array_equal(first, product(a, 2.0, 3.0, "again"))
        # new values in place, then in another array
        b = wl.Csr(a.rows, a.cols, a.row_ptr, a.col_ind, (a.values * dtype(-2.0)).astype(dtype), a.base, "new values")
        old = da.val
        other = hiprt.DeviceArray.from_numpy(b.values)
        da.val = other
        try:
            product(b, 2.0, 3.0, "other array")
        finally:
            da.val = old
            other.free()
        da.val.copy_from(b.values)
        product(b, 2.0, 3.0, "in place")
    finally:
        lib.alphasparse_dcu_destroy_mat_info(info)
        da.free()


@pytest.mark.parametrize("make", [lambda: wl.uniform_rows(20000, 20000, 10, np.float32), lambda: wl.uniform_rows(20000, 20000, 17, np.float64)],
                         ids=["f32", "f64"])
def test_without_a_check_the_copy_multiplies(gpu, make, monkeypatch):
    """ALSPARSE_AMD_VALUE_CHECK=off: nothing stands in front of the copy of A^T, whose multiply alone is the faster one.  The
    product has the bits of a multiply with the copy's own arrays; another value array still gives its own product."""
    monkeypatch.setenv("ALSPARSE_AMD_VALUE_CHECK", "off")
    a = make()
    x, y0 = wl.uniform(a.rows, a.dtype, 3), wl.uniform(a.cols, a.dtype, 4)
    lib, da, T = capi.load(), DeviceCsr(a), capi.scalar_type(a.dtype)
    plan, direct = c_void_p(), c_void_p()
    code = capi.dtype_tag(a.dtype)

    def product(p, op, arrays):
        ws = capi.Workspace(lib, p)
        dx, dy = hiprt.DeviceArray.from_numpy(x), hiprt.DeviceArray.from_numpy(y0)
        assert capi.plan_csrmv(lib, None, p, op, T(1.5), *arrays, dx.c_ptr(), T(0.5), dy.c_ptr(), ws) == 0
        hiprt.synchronize()
        y = dy.to_numpy()
        dx.free()
        dy.free()
        return y

    try:
        announce("transposed, values not checked", a.name)
        own = (da.val.c_ptr(), da.row_ptr.c_ptr(), da.col.c_ptr())
        assert lib.asamd_csr_plan_create_dtype(None, a.rows, a.cols, a.nnz, own[1], own[2], own[0], 0, code, 1, byref(plan)) == 0
        assert lib.asamd_csr_plan_build_transpose(None, plan, own[1], own[2], own[0]) == 0
        row, col, val = c_void_p(), c_void_p(), c_void_p()
        assert lib.asamd_csr_plan_transpose_arrays(plan, 0, byref(row), byref(col), byref(val)) == 0
        assert lib.asamd_csr_plan_create_dtype(None, a.cols, a.rows, a.nnz, row, col, val, 0, code, 1, byref(direct)) == 0
        y = product(plan, 1, own)
        check_trans(a, 1.5, x, 0.5, y0, y, "not checked")
        assert np.array_equal(y, product(direct, 0, (val, row, col)))
        b = wl.Csr(a.rows, a.cols, a.row_ptr, a.col_ind, (a.values * a.dtype.type(-2.0)).astype(a.dtype), 0, "other")
        other = hiprt.DeviceArray.from_numpy(b.values)
        check_trans(b, 1.5, x, 0.5, y0, product(plan, 1, (other.c_ptr(),) + own[1:]), "another array")
        da.val.copy_from(b.values)
        assert lib.asamd_csr_plan_refresh_values(None, plan, own[1], own[2], own[0]) == 0
        check_trans(b, 1.5, x, 0.5, y0, product(plan, 1, own), "refreshed")
        other.free()
    finally:
        if direct:
            lib.asamd_csr_plan_destroy(direct)
        lib.asamd_csr_plan_destroy(plan)
        da.free()
