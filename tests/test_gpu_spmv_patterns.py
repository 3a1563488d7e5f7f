"""SpMV with a pattern number per row instead of column numbers (asamd_patterns_build, asamd_spmv_patterns): rows whose
lists of distances (column - row) are one of at most 256.  Results are compared with the CPU oracle; matrices that the
layout must refuse leave it empty."""
from ctypes import addressof, byref, cast, c_void_p

import numpy as np
import pytest

from alsparse_amd import capi, hiprt, workloads as wl
from helpers import DeviceCsr, announce, check_spmv, run_csrmv

pytestmark = pytest.mark.gpu

DTYPES = {"f32": np.float32, "f64": np.float64, "c64": np.complex64}


def _vector(n, dtype, stream):
    return wl.complex_vector(n, dtype, stream) if np.dtype(dtype).kind == "c" else wl.uniform(n, dtype, stream)


def _check(a, alpha, x, beta, y0, y, what):
    """Real types against the oracle.  complex64 against 64-bit sums: a row of k entries is k complex fmas and the final
    scaling and addition, each of at most 2 * 2^-24 of what it adds up."""
    if np.dtype(a.dtype).kind != "c":
        check_spmv(a, alpha, x, beta, y0, y, what)
        return
    rp = a.row_ptr.astype(np.int64) - a.base
    prod = a.values.astype(np.complex128) * x.astype(np.complex128)[a.col_ind - a.base]
    ref = alpha * np.add.reduceat(prod, rp[:-1]) + beta * y0.astype(np.complex128)
    size = abs(alpha) * np.add.reduceat(np.abs(prod), rp[:-1]) + abs(beta) * np.abs(y0)
    assert np.all(np.abs(y - ref) <= 2 * 2.0 ** -24 * (np.diff(rp) + 4) * size), what


def _patterned(m, n, patterns, seed, dtype, base):
    """Row r has a random one of the patterns; its columns are r plus the pattern's distances, moved into [0, n)."""
    rng = np.random.default_rng(seed)
    rows = []
    for r in range(m):
        d = patterns[int(rng.integers(len(patterns)))]
        c = r + d
        rows.append(c - min(0, int(c.min())) - max(0, int(c.max()) - (n - 1)))
    row_ptr = np.zeros(m + 1, dtype=np.int64)
    np.cumsum([len(c) for c in rows], out=row_ptr[1:])
    col = np.concatenate(rows)
    return wl.Csr(m, n, (row_ptr + base).astype(np.int32), (col + base).astype(np.int32),
                  wl.uniform(int(row_ptr[-1]), dtype, 7, seed), base, "patterned")


def _group(a):
    cap, longest, g = 64 // a.dtype.itemsize, int(np.diff(a.row_ptr).max()), 1
    while g * cap < longest:
        g *= 2
    return g, longest


def _build(da):
    a, lib = da.a, capi.load()
    g, longest = _group(a)
    layout = capi.asamd_pattern_layout()
    assert lib.asamd_patterns_build(None, a.rows, a.nnz, a.base, g, longest, da.row_ptr.c_ptr(), da.col.c_ptr(),
                                    byref(layout)) == 0
    return layout


def _multiply(da, layout, alpha, x, beta, y0):
    a, lib = da.a, capi.load()
    T = capi.scalar_type(a.dtype)
    al, be = T(alpha), T(beta)
    dx, dy = hiprt.DeviceArray.from_numpy(x), hiprt.DeviceArray.from_numpy(y0)
    args = capi.asamd_spmv_args({"float32": 0, "float64": 1, "complex64": 2}[np.dtype(a.dtype).name], a.rows, a.cols, a.nnz, a.base,
                                cast(addressof(al), c_void_p), cast(addressof(be), c_void_p), da.val.c_ptr(),
                                da.row_ptr.c_ptr(), da.col.c_ptr(), dx.c_ptr(), dy.c_ptr())
    st = lib.asamd_spmv_patterns(None, byref(args), byref(layout))
    hiprt.synchronize()
    y = dy.to_numpy()
    dx.free()
    dy.free()
    return st, y


@pytest.mark.parametrize("name", list(DTYPES))
@pytest.mark.parametrize("base", [0, 1])
@pytest.mark.parametrize("longest", [1, 2, 5, 8, 9, 16, 17, 27, 64])
def test_row_lengths_across_the_lane_groups(gpu, name, base, longest):
    """Rows of 1 .. longest entries (every lane group and every unrolled length), blocks that start anywhere in a 128-bit
    piece, a last workgroup that ends inside the matrix and inside a piece."""
    rng = np.random.default_rng(longest)
    lengths = sorted({1, longest, (longest + 1) // 2, max(1, longest - 1)})
    patterns = [np.sort(rng.choice(np.arange(-200, 200), size=k, replace=False)) for k in lengths for _ in range(3)]
    a = _patterned(3001 + longest, 3300, patterns, longest + base, np.float64, base)
    # (rows moved at the matrix' borders have patterns of their own: keep those few)
    keep = slice(300, 300 + 2501 + longest % 5)
    rp = a.row_ptr[keep.start:keep.stop + 1].astype(np.int64)
    lo, hi = int(rp[0]) - base, int(rp[-1]) - base
    dtype = DTYPES[name]
    b = wl.Csr(keep.stop - keep.start, a.cols, (rp - lo).astype(np.int32), a.col_ind[lo:hi].copy(),
               _vector(hi - lo, dtype, 9), base, "patterned")
    x, y0 = _vector(b.cols, dtype, 3), _vector(b.rows, dtype, 4)
    da = DeviceCsr(b)
    layout = _build(da)
    try:
        assert layout.pid, "no layout for a dozen patterns"
        for alpha, beta in ((1.0, 0.0), (-1.5, 0.5)):
            announce("patterns:", name, "base", base, "longest", longest, alpha, beta)
            st, y = _multiply(da, layout, alpha, x, beta, y0)
            assert st == 0
            _check(b, alpha, x, beta, y0, y, "patterns %s" % ((alpha, beta),))
    finally:
        capi.load().asamd_patterns_free(byref(layout))
        da.free()


@pytest.mark.parametrize("longest", [3, 9, 27])
@pytest.mark.parametrize("rows", [1, 15, 16, 17, 31, 32, 63, 64, 65, 127, 128, 129, 255, 256, 257, 511, 513])
def test_matrices_that_end_around_a_wave(gpu, rows, longest):
    """A row's place among its wave's entries is the sum of the lengths before it: the last wave's rows begin or end there,
    waves without rows follow it."""
    patterns = [np.arange(k) * 3 for k in (longest, 1, longest - 1)]
    a = _patterned(rows + 100, rows + 300, patterns, rows, np.float64, 0)
    rp = a.row_ptr[:rows + 1].copy()
    rp_end = int(rp[-1])
    b = wl.Csr(rows, a.cols, rp, a.col_ind[:rp_end].copy(), a.values[:rp_end].copy(), 0, "patterned")
    x, y0 = wl.uniform(b.cols, b.dtype, 3), wl.uniform(b.rows, b.dtype, 4)
    da = DeviceCsr(b)
    layout = _build(da)
    try:
        assert layout.pid
        announce("patterns: rows", rows, "longest", longest)
        st, y = _multiply(da, layout, 1.5, x, 0.5, y0)
        assert st == 0
        _check(b, 1.5, x, 0.5, y0, y, "%d rows" % rows)
    finally:
        capi.load().asamd_patterns_free(byref(layout))
        da.free()


@pytest.mark.parametrize("name,longest,mbytes", [("f32", 5, 140), ("f32", 5, 160), ("f32", 27, 270), ("f32", 27, 300), ("f64", 5, 160),
                                                 ("f64", 27, 140), ("f64", 27, 160), ("f64", 27, 300), ("c64", 27, 200)])
def test_forms_on_both_sides_of_their_lines(gpu, name, longest, mbytes):
    """The form whose loads wait for as little as can be, up to 150 MB, the one whose values go first, and from 280 MB the one
    whose values bypass the caches: a last wave with a few rows in each."""
    dtype = DTYPES[name]
    size = np.dtype(dtype).itemsize
    mean = longest - 0.5  # rows of longest and longest - 1 entries
    m = int(mbytes * 1e6 / (mean * size + 5 + 2 * size)) // 256 * 256 + 7
    rng = np.random.default_rng(longest)
    which = rng.integers(0, 2, size=m)
    table = np.stack([np.arange(longest) * 3, np.arange(longest) * 3 + 1]).astype(np.int32)
    lengths = longest - which
    row_ptr = np.zeros(m + 1, dtype=np.int64)
    np.cumsum(lengths, out=row_ptr[1:])
    col = (np.arange(m, dtype=np.int32)[:, None] + table[which])[np.arange(longest)[None, :] < lengths[:, None]]
    a = wl.Csr(m, m + 3 * longest, row_ptr.astype(np.int32), col, _vector(col.size, dtype, 9), 0, "patterned")
    x, y0 = _vector(a.cols, dtype, 3), _vector(a.rows, dtype, 4)
    da = DeviceCsr(a)
    layout = _build(da)
    try:
        assert layout.pid
        announce("patterns by size", name, longest, mbytes)
        st, y = _multiply(da, layout, 1.5, x, 0.5, y0)
        assert st == 0
        _check(a, 1.5, x, 0.5, y0, y, "%s %d MB" % (name, mbytes))
    finally:
        capi.load().asamd_patterns_free(byref(layout))
        da.free()


@pytest.mark.parametrize("what", ["many patterns", "an empty row", "a long row"])
def test_matrices_without_the_layout(gpu, what):
    """More patterns than a byte can number, an empty row, rows of 65 entries: no layout, and no error."""
    rng = np.random.default_rng(1)
    m, n = 4000, 5000
    count, longest = (600, 4) if what == "many patterns" else (4, 65 if what == "a long row" else 4)
    patterns = [np.sort(rng.choice(np.arange(0, 900), size=longest, replace=False)) for _ in range(count)]
    a = _patterned(m, n, patterns, 2, np.float32, 0)
    if what == "an empty row":
        rp = a.row_ptr.copy()
        rp[101] = rp[100]  # row 100 loses its entries to row 101
        a = wl.Csr(m, n, rp, a.col_ind, a.values, 0, "patterned")
    da = DeviceCsr(a)
    layout = _build(da)
    try:
        assert not layout.pid and layout.device_bytes == 0
    finally:
        da.free()


@pytest.mark.parametrize("count", [250, 255, 256, 257])
def test_every_slot_of_the_table_is_used(gpu, count):
    """As many patterns as a byte can number have the layout whatever order they arrive in, one more never has: rows of
    two entries, the second `d` columns behind the first, every `d` from 1 to `count` (a row's first distance is 0)."""
    rng = np.random.default_rng(count)
    m = 20000
    d = np.concatenate([np.arange(1, count + 1), rng.integers(1, count + 1, size=m - count)])
    rng.shuffle(d)
    col = np.stack([np.arange(m), np.arange(m) + d], axis=1).astype(np.int32).reshape(-1)
    a = wl.Csr(m, m + count, (2 * np.arange(m + 1)).astype(np.int32), col, wl.uniform(2 * m, np.float64, 7), 0, "pairs")
    x, y0 = wl.uniform(a.cols, a.dtype, 3), wl.uniform(a.rows, a.dtype, 4)
    da = DeviceCsr(a)
    try:
        for attempt in range(8):
            announce("patterns:", count, "patterns, attempt", attempt)
            layout = _build(da)
            try:
                assert bool(layout.pid) == (count <= 256)
                if layout.pid:
                    st, y = _multiply(da, layout, 1.5, x, 0.5, y0)
                    assert st == 0
                    check_spmv(a, 1.5, x, 0.5, y0, y, "%d patterns" % count)
            finally:
                capi.load().asamd_patterns_free(byref(layout))
    finally:
        da.free()


@pytest.mark.parametrize("name,entries,short,long,every,want", [
    ("f32", 2000000, 5, 5, 1, True),
    ("f32", 1000000, 5, 5, 1, False),   # a launch's latency
    ("f32", 2000000, 2, 12, 10, False),  # 12 gathers for every row of 3 entries on average
    ("f32", 2000000, 3, 4, 4, True),
    ("f32", 2000000, 18, 24, 4, False),  # two lanes a row
    ("f64", 2000000, 1, 8, 9, False),
    ("f64", 2000000, 14, 24, 4, True),
    ("c64", 2000000, 3, 6, 4, True),
])
def test_uneven_rows_stay_with_the_columns(gpu, name, entries, short, long, every, want):
    """The analysis keeps patterns where the gathers of rows padded to the longest are worth it: rows of `short` entries,
    every `every`-th of `long`, all of two patterns."""
    lib, dtype = capi.load(), DTYPES[name]
    rows = int(entries * every / ((every - 1) * short + long)) if every > 1 else entries // long
    lengths = np.where(np.arange(rows) % every == 0, long, short)
    row_ptr = np.concatenate([[0], np.cumsum(lengths)])
    row = np.repeat(np.arange(rows), lengths)
    col = (row + 7 * (np.arange(row.size) - row_ptr[row])).astype(np.int32)
    a = wl.Csr(rows, rows + 7 * long, row_ptr.astype(np.int32), col, _vector(row.size, dtype, 9), 0, "uneven")
    x, y0 = _vector(a.cols, dtype, 3), _vector(a.rows, dtype, 4)
    da = DeviceCsr(a)
    descr, info = capi.make_descr(), capi.alphasparse_dcu_mat_info_t()
    assert lib.alphasparse_dcu_create_mat_info(byref(info)) == 0
    try:
        assert getattr(lib, "alphasparse_dcu_%s_csrmv_analysis" % capi.prefix(dtype))(
            gpu.h, 0, a.rows, a.cols, a.nnz, byref(descr), da.val.c_ptr(), da.row_ptr.c_ptr(), da.col.c_ptr(), info) == 0
        st = lib.asamd_analysis_stats(info).contents
        assert st.algo == capi.ASAMD_SPMV_STREAM
        announce("patterns: uneven rows", name, entries, short, long, every)
        assert (st.device_bytes >= a.rows) == want, "a byte per row with patterns, a constant without"
        assert st.row_patterns == want
        if want:  # (a family set from outside reads columns)
            for algo, patterns in ((capi.ASAMD_SPMV_STREAM, 0), (capi.ASAMD_SPMV_AUTO, 1)):
                assert lib.asamd_analysis_set_algo(info, algo) == 0
                assert lib.asamd_analysis_stats(info).contents.row_patterns == patterns
                _check(a, 1.5, x, 0.5, y0, run_csrmv(gpu, da, 1.5, x, 0.5, y0, info=info), "uneven rows")
        _check(a, 1.5, x, 0.5, y0, run_csrmv(gpu, da, 1.5, x, 0.5, y0, info=info), "uneven rows")
    finally:
        lib.alphasparse_dcu_destroy_mat_info(info)
        da.free()


def test_an_analysed_stencil_keeps_patterns_and_reads_the_callers_values(gpu):
    """27-point stencil of 45 x 44 x 43 points (2.1 M entries) through the public API: patterns instead of a copy, the
    values read in place (new ones need nothing), and a value array that is not 16-byte aligned still multiplies."""
    lib = capi.load()
    a = wl.stencil3d(45, 44, 43, np.float32)
    x, y0 = wl.uniform(a.cols, a.dtype, 3), wl.uniform(a.rows, a.dtype, 4)
    for shift in (0, 1):
        da = DeviceCsr(a, shift)
        descr = capi.make_descr(base=a.base)
        info = capi.alphasparse_dcu_mat_info_t()
        assert lib.alphasparse_dcu_create_mat_info(byref(info)) == 0
        try:
            assert lib.alphasparse_dcu_s_csrmv_analysis(gpu.h, 0, a.rows, a.cols, a.nnz, byref(descr), da.val.c_ptr(),
                                                        da.row_ptr.c_ptr(), da.col.c_ptr(), info) == 0
            st = lib.asamd_analysis_stats(info).contents
            assert st.algo == capi.ASAMD_SPMV_STREAM
            assert a.rows <= st.device_bytes < a.nnz, "a byte per row, and no copy"
            announce("patterns: analysed stencil, shift", shift)
            check_spmv(a, 1.5, x, 0.5, y0, run_csrmv(gpu, da, 1.5, x, 0.5, y0, info=info), "stencil")
            if shift == 0:
                b = wl.Csr(a.rows, a.cols, a.row_ptr, a.col_ind, wl.uniform(a.nnz, a.dtype, 21), a.base, a.name)
                da.val.copy_from(b.values)
                check_spmv(b, 1.0, x, 0.0, y0, run_csrmv(gpu, da, 1.0, x, 0.0, y0, info=info), "new values in place")
        finally:
            lib.alphasparse_dcu_destroy_mat_info(info)
            da.free()
