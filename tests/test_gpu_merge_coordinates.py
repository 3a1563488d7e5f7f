"""Merge-path without a table of coordinates: every workgroup finds its own two, 64 probes at a time.  Compared with the
CPU oracle at one workgroup, at the edges of two and three, and with runs of empty rows and rows longer than workgroups."""
from ctypes import byref, c_void_p, cast

import numpy as np
import pytest

from alsparse_amd import capi, hiprt, workloads as wl
from helpers import DeviceCsr, announce, check_spmv, run_plan_csrmv
from helpers_shapes import csr_from_lengths

pytestmark = pytest.mark.gpu

LENGTHS = {
    "one workgroup": [3] * 100,
    "edge of two": [1] * 1024,            # rows + entries: exactly two workgroups of 1 024 items, one of eight per thread
    "one item more": [1] * 1024 + [0],
    "one item less": [1] * 1023 + [0],
    "edge of four": [1] * 2048,           # the same for 2 048 items
    "one item past four": [1] * 2048 + [0],
    "65 rows": [0] * 64 + [5000],
    "empty runs": [0] * 3000 + [7000] + [0] * 5000 + [1, 0, 2, 4096, 0] * 3 + [0] * 2000,
    "nothing but a long row": [20000],
    "skewed": [int(30000 / (i + 1)) for i in range(4000)],
}


@pytest.mark.parametrize("dtype,items", [(np.float32, None), (np.float64, None), (np.float32, 8)], ids=["f32", "f64", "f32_8"])
@pytest.mark.parametrize("base", [0, 1])
@pytest.mark.parametrize("shape", list(LENGTHS))
def test_workgroups_find_their_coordinates(gpu, shape, base, dtype, items, monkeypatch):
    """items: per thread; 4-byte values take eight, in workgroups of 2 048, where they are more than 2^25."""
    if items:
        monkeypatch.setenv("ALSPARSE_AMD_MERGE_IPT", str(items))
    a = csr_from_lengths(LENGTHS[shape], 30000, dtype, base=base)
    x, y0 = wl.uniform(a.cols, dtype, 3), wl.uniform(a.rows, dtype, 4)
    da = DeviceCsr(a)
    try:
        for alpha, beta in ((1.0, 0.0), (-1.5, 0.5)):
            announce("merge coordinates", shape, np.dtype(dtype).name, "base", base, alpha, beta)
            y = run_plan_csrmv(da, "merge", alpha, x, beta, y0, trusted=0)
            check_spmv(a, alpha, x, beta, y0, y, shape)
            # the same sums in the same order with the table that an analysis makes
            assert np.array_equal(y, run_plan_csrmv(da, "merge", alpha, x, beta, y0, trusted=1))
    finally:
        da.free()


@pytest.mark.parametrize("dtype,rows,alone", [(np.float32, 4096 * 64 - 64, True), (np.float32, 4096 * 64 + 64, True),
                                              (np.float32, 6144 * 64, True), (np.float32, 6144 * 64 + 1, False),
                                              (np.float64, 4096 * 64, True), (np.float64, 4096 * 64 + 1, False)])
def test_how_many_workgroups_need_no_table(gpu, dtype, rows, alone):
    """Scratch for the carries and nothing else: with it the merge path runs where its workgroups find their coordinates, the
    same bits as behind an analysis, and where they take a table a lane group per row runs in its place."""
    a = wl.uniform_rows(rows, 5000, 15, dtype)  # 16 items a row, 64 rows a workgroup of 1 024 items
    x, y0 = wl.uniform(a.cols, dtype, 3), wl.uniform(a.rows, dtype, 4)
    lib, T = capi.load(), capi.scalar_type(dtype)
    blocks, vs = (16 * rows + 1023) // 1024, np.dtype(dtype).itemsize
    room = -(-blocks * 4 // 256) * 256 + 2 * (-(-blocks * vs // 256) * 256)
    da, plan = DeviceCsr(a), c_void_p()
    ws, dx, dy = hiprt.DeviceArray((room,), np.uint8), hiprt.DeviceArray.from_numpy(x), hiprt.DeviceArray.from_numpy(y0)
    alpha, beta = T(1.5), T(0.5)
    try:
        assert lib.asamd_csr_plan_create(None, a.rows, a.cols, a.nnz, da.row_ptr.c_ptr(), da.col.c_ptr(), da.val.c_ptr(), 0, vs,
                                         0, byref(plan)) == 0
        assert lib.asamd_csr_plan_set_algo(plan, capi.ASAMD_SPMV_MERGE) == 0
        announce("merge without a table", rows, np.dtype(dtype).name)
        assert lib.asamd_csr_plan_csrmv(None, plan, 0, cast(byref(alpha), c_void_p), da.val.c_ptr(), da.row_ptr.c_ptr(),
                                        da.col.c_ptr(), dx.c_ptr(), cast(byref(beta), c_void_p), dy.c_ptr(), ws.c_ptr(), room) == 0
        hiprt.synchronize()
        y = dy.to_numpy()
        check_spmv(a, 1.5, x, 0.5, y0, y, "%d rows" % rows)
        assert np.array_equal(y, run_plan_csrmv(da, "merge" if alone else "vector", 1.5, x, 0.5, y0, trusted=1))
        assert not np.array_equal(y, run_plan_csrmv(da, "vector" if alone else "merge", 1.5, x, 0.5, y0, trusted=1))
    finally:
        if plan:
            lib.asamd_csr_plan_destroy(plan)
        for d in (ws, dx, dy, da):
            d.free()
