"""Row-sum tiles (spmv_sums.hpp): AUTO's multiply of an analysed matrix whose rows meet the same column blocks again and
again.  The reference has one kernel for every structure (src/kernel/dcu/level2/mv/csrmv/dcu_gemv_vector.h:14-57).

The tolerance is the textbook bound of a sum of L products in any order, gamma = (L + 4) u per row, against the sum of the
absolute products in 64 bits (complex products: four roundings each, so twice that)."""
from ctypes import addressof, byref, c_void_p, cast

import numpy as np
import pytest
import scipy.sparse as sp

from alsparse_amd import capi, hiprt, workloads as wl
from helpers import ALGOS, DeviceCsr, announce

pytestmark = pytest.mark.gpu

DTYPES = [np.float32, np.float64, np.complex64, np.complex128]


def _numbers(rng, n, dtype):
    v = rng.uniform(-1, 1, n)
    return (v + 1j * rng.uniform(-1, 1, n) if np.dtype(dtype).kind == "c" else v).astype(dtype)


def _matrix(lengths, n, dtype, seed, base=0, crowd=3, shuffled=False):
    """Rows of the given lengths, columns crowding towards 0 (repeats stay), ascending or in any order."""
    rng = np.random.default_rng(seed)
    lengths = np.asarray(lengths, dtype=np.int64)
    m = lengths.size
    row_ptr = np.concatenate([[0], np.cumsum(lengths)])
    row = np.repeat(np.arange(m), lengths)
    col = np.minimum((n * rng.random(row_ptr[-1]) ** crowd).astype(np.int64), n - 1)
    if not shuffled:
        col = np.sort(row * n + col) % n
    a = wl.Csr(m, n, (row_ptr + base).astype(np.int32), (col + base).astype(np.int32),
               _numbers(rng, row_ptr[-1], dtype), base, "rows %d cols %d" % (m, n))
    return a


def _check(a, alpha, x, beta, y0, y, what=""):
    wide = np.complex128 if np.iscomplexobj(a.values) else np.float64
    col, ptr = a.col_ind - a.base, a.row_ptr - a.base
    A = sp.csr_matrix((a.values.astype(wide), col, ptr), shape=(a.rows, a.cols))
    ref = alpha * (A @ x.astype(wide)) + beta * y0.astype(wide)
    B = sp.csr_matrix((np.abs(a.values).astype(np.float64), col, ptr), shape=(a.rows, a.cols))
    size = abs(alpha) * (B @ np.abs(x).astype(np.float64)) + abs(beta) * np.abs(y0)
    u = np.finfo(a.dtype).eps / 2
    bound = (np.diff(ptr) + 4) * u * (2 if np.iscomplexobj(a.values) else 1) * size
    off = np.abs(y - ref) - bound
    assert (off <= 0).all(), "%s: row %d off by %.3e, allowed %.3e" % (what, off.argmax(), off.max() + bound[off.argmax()],
                                                                      bound[off.argmax()])


class Plan:
    def __init__(self, a, trusted):
        self.lib, self.da, self.plan = capi.load(), DeviceCsr(a), c_void_p()
        assert self.lib.asamd_csr_plan_create_dtype(None, a.rows, a.cols, a.nnz, self.da.row_ptr.c_ptr(), self.da.col.c_ptr(),
                                                    self.da.val.c_ptr(), a.base, capi.dtype_tag(a.dtype), trusted,
                                                    byref(self.plan)) == 0
        self.stats = self.lib.asamd_csr_plan_stats(self.plan).contents
        self.ws = capi.Workspace(self.lib, self.plan)

    def multiply(self, alpha, x, beta, y0, val=None, ws=None, op=0):
        T = capi.scalar_type(self.da.a.dtype)
        dx, dy = hiprt.DeviceArray.from_numpy(x), hiprt.DeviceArray.from_numpy(y0)
        assert capi.plan_csrmv(self.lib, None, self.plan, op, T(alpha), (val or self.da.val).c_ptr(), self.da.row_ptr.c_ptr(),
                               self.da.col.c_ptr(), dx.c_ptr(), T(beta), dy.c_ptr(), ws or self.ws) == 0
        hiprt.synchronize()
        y = dy.to_numpy()
        dx.free()
        dy.free()
        return y

    def close(self):
        self.lib.asamd_csr_plan_destroy(self.plan)
        self.da.free()


def _tail(m, seed, longest):
    rng = np.random.default_rng(seed)
    lengths = np.minimum((1 / rng.random(m)).astype(np.int64), longest)
    lengths[rng.random(m) < 0.1] = 0
    return lengths


def _width(dtype):
    return 131072 // np.dtype(dtype).itemsize  # columns of a column block


# structures whose choice from the row lengths alone is merge-path, so that a forced analysis lays out the tiles
SHAPES = {
    "one_block": lambda d: _matrix(_tail(70001, 1, 100), 100, d, 1),
    "block_edge": lambda d: _matrix(_tail(30000, 2, 9000), _width(d), d, 2),
    "past_the_edge": lambda d: _matrix(_tail(30000, 3, 9000), _width(d) + 1, d, 3, crowd=1),
    # hub rows that fill whole spans (2048 entries) of one column block, beside short ones
    "hubs": lambda d: _matrix([60000] * 3 + [0] * 61 + list(_tail(5000, 4, 50)), 70000, d, 4, crowd=6),
    "only_long_rows": lambda d: _matrix([5000] * 100, 50000, d, 5, crowd=1),
    # rows of exactly one and two spans, one entry more and one less
    "span_edges": lambda d: _matrix([2047, 2048, 2049, 4096, 1, 0, 1024, 1023, 1025] * 10 + [3] * 2000, 3000, d, 6, crowd=1),
    "unsorted_base_one": lambda d: _matrix(_tail(40000, 7, 4000), 2 * _width(d) + 77, d, 7, base=1, shuffled=True),
    # column blocks of many and of few spans, cut into pieces that are not all equally long
    "uneven_pieces": lambda d: _matrix(_tail(150001, 10, 3000), 5 * _width(d) + 11, d, 10),
    # taller than a row block: several of them, the last one short
    "many_rows": lambda d: _matrix(_tail(700001, 8, 3000), 40000, d, 8),
}


@pytest.mark.parametrize("dtype", DTYPES, ids=["f32", "f64", "c64", "c128"])
@pytest.mark.parametrize("shape", sorted(SHAPES))
def test_edges_against_64_bits(gpu, shape, dtype):
    a = SHAPES[shape](dtype)
    rng = np.random.default_rng(9)
    x, y0 = _numbers(rng, a.cols, dtype), _numbers(rng, a.rows, dtype)
    p = Plan(a, 2)
    try:
        announce("row sums", shape, np.dtype(dtype).name)
        assert p.stats.row_sums == 1 and p.stats.algo == capi.ASAMD_SPMV_MERGE
        for alpha, beta in ((1.0, 0.0), (-1.5, 0.5)):
            y = p.multiply(alpha, x, beta, y0)
            _check(a, alpha, x, beta, y0, y, shape)
            assert np.array_equal(y, p.multiply(alpha, x, beta, y0)), "the same bits on every run"
    finally:
        p.close()


@pytest.mark.parametrize("dtype", DTYPES, ids=["f32", "f64", "c64", "c128"])
@pytest.mark.parametrize("shape", ["past_the_edge", "hubs", "span_edges", "uneven_pieces"])
def test_every_form_of_the_first_phase(gpu, shape, dtype):
    """Loads and stores through the memory-side cache or past it, which the layout's size decides otherwise (256 MB of streams
    and sums, 512 MB of sums): one sum per row and column block, the same bits in all three."""
    a = SHAPES[shape](dtype)
    rng = np.random.default_rng(21)
    x, y0 = _numbers(rng, a.cols, dtype), _numbers(rng, a.rows, dtype)
    lib, T, layout, da = capi.load(), capi.scalar_type(dtype), capi.asamd_sums_layout(), DeviceCsr(a)
    alpha, beta = T(-1.5), T(0.5)
    dx, dy, sums = hiprt.DeviceArray.from_numpy(x), hiprt.DeviceArray.from_numpy(y0), None
    try:
        assert lib.asamd_sums_build(None, capi.dtype_tag(a.dtype), a.rows, a.cols, a.nnz, a.base, da.row_ptr.c_ptr(),
                                    da.col.c_ptr(), da.val.c_ptr(), a.nnz, byref(layout)) == 0
        assert layout.tval and layout.nnz == a.nnz and 0 < layout.sums <= a.nnz
        sums = hiprt.DeviceArray((layout.sums,), a.dtype)
        args = capi.asamd_spmv_args(capi.dtype_tag(a.dtype), a.rows, a.cols, a.nnz, a.base, cast(addressof(alpha), c_void_p),
                                    cast(addressof(beta), c_void_p), da.val.c_ptr(), da.row_ptr.c_ptr(), da.col.c_ptr(),
                                    dx.c_ptr(), dy.c_ptr())
        got = []
        for form in (-1, 0, 1, 2):
            announce("row sums, form", form, shape, np.dtype(dtype).name)
            dy.copy_from(y0)
            assert lib.asamd_spmv_sums_form(None, byref(args), byref(layout), sums.c_ptr(), None, form) == 0
            hiprt.synchronize()
            got.append(dy.to_numpy())
        _check(a, -1.5, x, 0.5, y0, got[0], shape)
        for y in got[1:]:
            assert np.array_equal(y, got[0])
        for form in (-2, 3):
            assert lib.asamd_spmv_sums_form(None, byref(args), byref(layout), sums.c_ptr(), None, form) == 1
    finally:
        lib.asamd_sums_free(byref(layout))
        for d in (dx, dy, sums, da):
            if d:
                d.free()


def test_slots_without_an_entry_leave_nothing_behind(gpu):
    """Spans end in slots that name column 0 with value zero: an infinite or NaN x[0] reaches only the rows that hold
    column 0, and beta == 0 does not read y."""
    a = _matrix(_tail(40000, 11, 5000), 90000, np.float32, 11)
    a.col_ind[a.col_ind == 0] = 1
    rng = np.random.default_rng(12)
    x, y0 = _numbers(rng, a.cols, np.float32), np.full(a.rows, np.nan, np.float32)
    p = Plan(a, 2)
    try:
        announce("row sums, x[0] not finite")
        assert p.stats.row_sums == 1
        for bad in (np.inf, np.nan):
            x[0] = bad
            y = p.multiply(1.0, x, 0.0, y0)
            assert np.isfinite(y).all()
    finally:
        p.close()


def test_values_follow_the_caller(gpu):
    """Values rewritten in place are picked up; another value array, a family set from outside and a workspace without room
    take the family that the analysis chose."""
    a = _matrix(_tail(50000, 13, 20000), 200000, np.float64, 13)
    rng = np.random.default_rng(14)
    x, y0 = _numbers(rng, a.cols, np.float64), _numbers(rng, a.rows, np.float64)
    p = Plan(a, 2)
    try:
        announce("row sums, values")
        assert p.stats.row_sums == 1
        first = p.multiply(1.0, x, 0.5, y0)
        other = wl.Csr(a.rows, a.cols, a.row_ptr, a.col_ind, _numbers(rng, a.nnz, np.float64), 0, "other")
        d_other = hiprt.DeviceArray.from_numpy(other.values)
        _check(other, 1.0, x, 0.5, y0, p.multiply(1.0, x, 0.5, y0, val=d_other), "another array")
        p.da.val.copy_from(other.values)
        second = p.multiply(1.0, x, 0.5, y0)
        _check(other, 1.0, x, 0.5, y0, second, "in place")
        p.da.val.copy_from(a.values)
        assert np.array_equal(p.multiply(1.0, x, 0.5, y0), first)
        small = capi.Workspace(p.lib, p.plan)
        small.bytes = 4096
        _check(a, 1.0, x, 0.5, y0, p.multiply(1.0, x, 0.5, y0, ws=small), "no room")
        assert p.lib.asamd_csr_plan_set_algo(p.plan, ALGOS["merge"]) == 0
        assert p.stats.row_sums == 0, "a family set from outside runs, not the tiles"
        _check(a, 1.0, x, 0.5, y0, p.multiply(1.0, x, 0.5, y0), "merge-path set from outside")
        assert p.lib.asamd_csr_plan_set_algo(p.plan, capi.ASAMD_SPMV_AUTO) == 0
        assert p.stats.row_sums == 1
        assert np.array_equal(p.multiply(1.0, x, 0.5, y0), first)
        d_other.free()
    finally:
        p.close()


def test_without_a_check_a_refresh_brings_the_values(gpu, monkeypatch):
    """ALSPARSE_AMD_VALUE_CHECK=off: the caller refreshes by hand, the tiles' values too."""
    monkeypatch.setenv("ALSPARSE_AMD_VALUE_CHECK", "off")
    a = _matrix(_tail(50000, 13, 20000), 200000, np.float64, 13)
    rng = np.random.default_rng(20)
    x, y0 = _numbers(rng, a.cols, np.float64), _numbers(rng, a.rows, np.float64)
    p = Plan(a, 2)
    try:
        announce("row sums, no check")
        assert p.stats.row_sums == 1 and p.stats.value_check == 0
        _check(a, 1.0, x, 0.5, y0, p.multiply(1.0, x, 0.5, y0), "values of the analysis")
        b = wl.Csr(a.rows, a.cols, a.row_ptr, a.col_ind, _numbers(rng, a.nnz, np.float64), 0, "new")
        p.da.val.copy_from(b.values)
        assert p.lib.asamd_csr_plan_refresh_values(None, p.plan, p.da.row_ptr.c_ptr(), p.da.col.c_ptr(), p.da.val.c_ptr()) == 0
        _check(b, 1.0, x, 0.5, y0, p.multiply(1.0, x, 0.5, y0), "refreshed")
    finally:
        p.close()


def test_single_values_poked_into_a_graph_count(gpu):
    """Merge-path and the hot-column kernel read csr_val on every multiply; the tiles that stand in for them hold a copy of
    it, 92 MB here, of which the usual check reads a quarter: one changed value anywhere has to show in the next product
    all the same."""
    a = wl.powerlaw_rmat(21, 50000, np.float32)
    lib = capi.load()
    assert int(lib.asamd_value_guard_run(a.nnz * 4)) >= 1024, "an array of which the usual check reads a part"
    rng = np.random.default_rng(17)
    x = wl.uniform(a.cols, a.dtype, 3)
    x[np.abs(x) < 0.1] = 0.5
    y0 = np.zeros(a.rows, np.float32)
    p = Plan(a, 1)
    try:
        announce("row sums, single values poked")
        assert p.stats.row_sums == 1 and p.stats.value_check == 1
        assert p.stats.algo in (capi.ASAMD_SPMV_MERGE, capi.ASAMD_SPMV_MERGE_HOT)
        vals = a.values.copy()
        p.multiply(1.0, x, 0.0, y0)
        for k in list(rng.integers(0, a.nnz, 8)) + [a.nnz - 1, 0]:
            vals[k] = np.float32(1000.0)
            p.da.val.copy_from(vals)
            b = wl.Csr(a.rows, a.cols, a.row_ptr, a.col_ind, vals, a.base, "poked")
            _check(b, 1.0, x, 0.0, y0, p.multiply(1.0, x, 0.0, y0), "value %d poked" % k)
    finally:
        p.close()


@pytest.mark.parametrize("name,make,want", [
    # rows of 16, and uneven rows of 30 on average, over 4 MB of x; matrices whose x the LDS or the caches hold stay as they are
    ("uniform", lambda: wl.uniform_rows(1 << 20, 1 << 20, 16, np.float32), 1),
    ("uneven", lambda: _matrix(np.random.default_rng(15).geometric(1 / 30, 700000), 1 << 20, np.float32, 15, crowd=1), 1),
    ("few_columns", lambda: wl.uniform_rows(1 << 20, 1 << 14, 8, np.float32), 0),
    ("stencil", lambda: wl.laplace2d(1500, 1400, np.float64), 0),
], ids=["uniform", "uneven", "few_columns", "stencil"])
def test_the_analysis_lays_them_out_where_they_pay(gpu, name, make, want, monkeypatch):
    a = make()
    rng = np.random.default_rng(16)
    x, y0 = _numbers(rng, a.cols, a.dtype), _numbers(rng, a.rows, a.dtype)
    p = Plan(a, 1)
    monkeypatch.setenv("ALSPARSE_AMD_ROW_SUMS", "0")
    q = Plan(a, 1)
    try:
        announce("row sums, analysis", name)
        assert p.stats.row_sums == want and q.stats.row_sums == 0
        assert p.stats.algo == q.stats.algo, "the family is the same with them and without"
        _check(a, 1.5, x, 0.5, y0, p.multiply(1.5, x, 0.5, y0), name)
        _check(a, 1.5, x, 0.5, y0, q.multiply(1.5, x, 0.5, y0), name + " without")
    finally:
        p.close()
        q.close()


@pytest.mark.parametrize("pick,algo", [("tiled", capi.ASAMD_SPMV_TILED), ("ell", capi.ASAMD_SPMV_ELL), ("base", None)])
@pytest.mark.parametrize("tune", ["model", "timed"])
def test_a_family_picked_for_the_analysis_is_the_one_that_runs(gpu, pick, algo, tune, monkeypatch):
    """ALSPARSE_AMD_TUNE_PICK overrides the analysis' verdict: the tiles do not take the picked family's place."""
    a = wl.uniform_rows(1 << 21, 1 << 21, 16, np.float32)
    monkeypatch.setenv("ALSPARSE_AMD_TUNE", tune)
    monkeypatch.setenv("ALSPARSE_AMD_TUNE_PICK", pick)
    p = Plan(a, 1)
    try:
        announce("row sums, picked", pick, tune)
        assert p.stats.row_sums == 0
        if tune == "model":  # (a timing run picks among the copies that it found worth laying out)
            assert p.stats.algo == algo if algo is not None else p.stats.tiled_built + p.stats.ell_built == 0
    finally:
        p.close()


@pytest.mark.parametrize("make", [lambda: wl.uniform_rows(1 << 21, 1 << 21, 16, np.float32),
                                  lambda: wl.powerlaw_rmat(21, 50000, np.float32)], ids=["uniform", "powerlaw"])
def test_a_timed_analysis_times_them(gpu, make, monkeypatch):
    """ALSPARSE_AMD_TUNE=timed: no estimate puts a kernel that was not timed in the place of the family that won."""
    a = make()
    rng = np.random.default_rng(18)
    x, y0 = _numbers(rng, a.cols, a.dtype), _numbers(rng, a.rows, a.dtype)
    q = Plan(a, 1)
    monkeypatch.setenv("ALSPARSE_AMD_TUNE", "timed")
    p = Plan(a, 1)
    try:
        announce("row sums, timed analysis")
        assert q.stats.row_sums == 1 and q.stats.tune_ms_sums > 0
        assert p.stats.tune_mode == 0 and p.stats.tune_ms_sums > 0 and p.stats.tune_ms_sums != q.stats.tune_ms_sums
        assert 0.5 * p.stats.tune_ms_sums < q.stats.tune_ms_sums < 2 * p.stats.tune_ms_sums
        _check(a, 1.5, x, 0.5, y0, p.multiply(1.5, x, 0.5, y0), "timed")
        y = p.multiply(1.5, x, 0.5, y0)
        assert np.array_equal(y, q.multiply(1.5, x, 0.5, y0)) == (p.stats.row_sums == 1)
    finally:
        p.close()
        q.close()


def _transposed(a, op):
    t = sp.csr_matrix((a.values if op == 1 else a.values.conj(), a.col_ind, a.row_ptr), shape=(a.rows, a.cols)).T.tocsr()
    return wl.Csr(a.cols, a.rows, t.indptr.astype(np.int32), t.indices.astype(np.int32), t.data, 0, "op %d" % op)


@pytest.mark.parametrize("dtype,op,m,n", [(np.float32, 1, 1 << 21, 1 << 21), (np.float64, 1, 1000003, 786433),
                                          (np.complex64, 2, 1000003, 786433)], ids=["f32_T", "f64_T", "c64_H"])
def test_the_copy_of_the_transpose_runs_on_them(gpu, dtype, op, m, n):
    """The copy of A^T (A^H) with row-sum tiles: its family's own copy is not laid out beside them, values rewritten in place
    are picked up, and a refresh takes another array."""
    a = wl.uniform_rows(m, n, 16, np.float64)
    rng = np.random.default_rng(19)
    a = wl.Csr(a.rows, a.cols, a.row_ptr, a.col_ind, _numbers(rng, a.nnz, dtype), 0, a.name)
    x, y0 = _numbers(rng, a.rows, dtype), _numbers(rng, a.cols, dtype)
    p = Plan(a, 1)
    try:
        announce("row sums of the transpose", np.dtype(dtype).name, op)
        build = p.lib.asamd_csr_plan_build_transpose if op == 1 else p.lib.asamd_csr_plan_build_conj_transpose
        assert build(None, p.plan, p.da.row_ptr.c_ptr(), p.da.col.c_ptr(), p.da.val.c_ptr()) == 0
        p.ws = capi.Workspace(p.lib, p.plan)
        st = p.lib.asamd_csr_plan_transpose_stats(p.plan).contents
        assert st.row_sums == 1 and p.stats.value_check == 1
        assert st.tiled_built + st.ell_built + st.hot_built + st.binned_built + st.xlds_slices == 0
        first = p.multiply(1.5, x, 0.5, y0, op=op)
        _check(_transposed(a, op), 1.5, x, 0.5, y0, first, "values of the analysis")
        assert np.array_equal(first, p.multiply(1.5, x, 0.5, y0, op=op))
        b = wl.Csr(a.rows, a.cols, a.row_ptr, a.col_ind, _numbers(rng, a.nnz, dtype), 0, "other values")
        p.da.val.copy_from(b.values)
        t = _transposed(b, op)
        second = p.multiply(1.5, x, 0.5, y0, op=op)
        _check(t, 1.5, x, 0.5, y0, second, "in place")
        small = capi.Workspace(p.lib, p.plan)
        small.bytes = 1 << 20  # the check of the values and no room for the sums
        _check(t, 1.5, x, 0.5, y0, p.multiply(1.5, x, 0.5, y0, op=op, ws=small), "no room")
        d_other = hiprt.DeviceArray.from_numpy(a.values)
        p.da.val.copy_from(np.zeros_like(a.values))
        assert p.lib.asamd_csr_plan_refresh_values(None, p.plan, p.da.row_ptr.c_ptr(), p.da.col.c_ptr(), d_other.c_ptr()) == 0
        assert np.array_equal(first, p.multiply(1.5, x, 0.5, y0, op=op, val=d_other)), "refreshed from another array"
        _check(a, 1.5, y0, 0.5, x, p.multiply(1.5, y0, 0.5, x, val=d_other), "the product with A, refreshed")
        d_other.copy_from(b.values)
        assert np.array_equal(second, p.multiply(1.5, x, 0.5, y0, op=op, val=d_other)), "in place in the array of the refresh"
        d_other.free()
    finally:
        p.close()
