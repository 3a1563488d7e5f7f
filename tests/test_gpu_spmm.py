"""GPU parity of CSR SpMM against the CPU oracle, through alphasparse_dcu_?_csrmm.
Tolerance per element as for SpMV (1e-4 fp32 / 1e-12 fp64)."""
from ctypes import byref

import numpy as np
import pytest

from alsparse_amd import capi, hiprt, workloads as wl
from oracle import oracle as orc
from helpers import TOL, DeviceCsr, announce
from helpers_shapes import csr_from_lengths

pytestmark = pytest.mark.gpu


def run_csrmm(h, da, layout, trans_b, alpha, B, ldb, beta, C0, ldc, n, k):
    a = da.a
    lib = capi.load()
    T = capi.scalar_type(a.dtype)
    descr = capi.make_descr(base=a.base)
    dB, dC = hiprt.DeviceArray.from_numpy(B), hiprt.DeviceArray.from_numpy(C0)
    al, be = T(alpha), T(beta)
    st = getattr(lib, "alphasparse_dcu_%s_csrmm" % capi.prefix(a.dtype))(
        h.h, 0, trans_b, layout, a.rows, n, k, a.nnz, byref(al), byref(descr), da.val.c_ptr(), da.row_ptr.c_ptr(),
        da.col.c_ptr(), dB.c_ptr(), ldb, byref(be), dC.c_ptr(), ldc)
    assert st == 0, "csrmm status %d" % st
    hiprt.synchronize()
    out = dC.to_numpy()
    dB.free()
    dC.free()
    return out


def check(a, alpha, B2, beta, C02, C2, what):
    ref = orc.csrmm_plain(a, alpha, np.ascontiguousarray(B2), beta, np.ascontiguousarray(C02))
    err = orc.csrmm_err(a, alpha, np.ascontiguousarray(B2), beta, np.ascontiguousarray(C02), np.ascontiguousarray(C2), ref)
    assert err.zero_den_mismatch == 0, what
    assert err.full <= TOL[a.dtype], "%s: %r" % (what, err)
    if beta == 0:
        assert err.strict <= TOL[a.dtype], "%s: %r" % (what, err)


MATS = {
    "uniform32": lambda dt, base: wl.uniform_rows(3000, 2500, 32, dt, base=base),
    "powerlaw": lambda dt, base: wl.powerlaw_rmat(11, 1500, dt, base=base),
    "ragged": lambda dt, base: csr_from_lengths([0, 1, 0, 130, 64, 65, 63, 2, 0, 300, 1, 1], 400, dt, base=base),
}


@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
@pytest.mark.parametrize("mat", sorted(MATS))
@pytest.mark.parametrize("n", [1, 2, 3, 7, 16, 17, 24, 31, 32, 64, 100, 128, 300])
def test_row_major(gpu, mat, n, dtype):
    for base in (0, 1):
        a = MATS[mat](dtype, base)
        da = DeviceCsr(a)
        try:
            for pad_b, pad_c in ((0, 0), (3, 5)):
                ldb, ldc = n + pad_b, n + pad_c
                Bfull = wl.uniform(a.cols * ldb, dtype, 5).reshape(a.cols, ldb)
                Cfull = wl.uniform(a.rows * ldc, dtype, 4).reshape(a.rows, ldc)
                for alpha, beta in ((1.5, 0.5), (1.0, 0.0)):
                    announce("spmm row-major", mat, n, np.dtype(dtype).name, base, ldb, ldc, alpha, beta)
                    out = run_csrmm(gpu, da, capi.ALPHA_SPARSE_LAYOUT_ROW_MAJOR, 0, alpha, Bfull, ldb, beta, Cfull, ldc, n, a.cols)
                    check(a, alpha, Bfull[:, :n], beta, Cfull[:, :n], out[:, :n], "%s n=%d" % (mat, n))
                    assert np.array_equal(out[:, n:], Cfull[:, n:]), "padding columns of C were touched"
        finally:
            da.free()


@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
@pytest.mark.parametrize("seed", range(12))
def test_random_structures_widths_and_layouts(gpu, seed, dtype):
    """Seeded random structures (row-length law, base), a random number of dense columns and random padding of the
    leading dimensions, row-major and column-major."""
    rng = np.random.default_rng(500 + seed)
    m, cols = int(rng.integers(1, 1500)), int(rng.integers(1, 2000))
    law = int(rng.integers(0, 4))
    if law == 0:
        lengths = np.full(m, int(rng.integers(1, 40)))
    elif law == 1:
        lengths = rng.integers(0, int(rng.integers(2, 120)) + 1, size=m)
    elif law == 2:
        lengths = rng.geometric(1.0 / float(rng.integers(2, 20)), size=m) - 1
    else:
        lengths = rng.integers(0, 5, size=m)
        lengths[rng.integers(0, m, size=max(1, m // 100))] = int(rng.integers(200, 1500))
    base = int(rng.integers(0, 2))
    a = csr_from_lengths(list(np.minimum(lengths, cols)), cols, dtype, seed=int(rng.integers(1, 1 << 30)), base=base)
    if a.nnz == 0:
        pytest.skip("drew a matrix without entries")
    n = int(rng.choice([1, 2, 3, 4, 5, 8, 12, 16, 17, 20, 31, 32, 33, 48, 64, 65, 96, 128, 130]))
    da = DeviceCsr(a)
    try:
        ldb, ldc = n + int(rng.integers(0, 4)), n + int(rng.integers(0, 4))
        B = wl.uniform(a.cols * ldb, dtype, 5).reshape(a.cols, ldb)
        C0 = wl.uniform(a.rows * ldc, dtype, 4).reshape(a.rows, ldc)
        alpha, beta = ((1.5, 0.5), (1.0, 0.0), (-2.0, 1.0))[int(rng.integers(0, 3))]
        announce("spmm random structure, row-major", seed, a.name, n, np.dtype(dtype).name, base, ldb, ldc, alpha, beta)
        out = run_csrmm(gpu, da, capi.ALPHA_SPARSE_LAYOUT_ROW_MAJOR, 0, alpha, B, ldb, beta, C0, ldc, n, a.cols)
        check(a, alpha, B[:, :n], beta, C0[:, :n], out[:, :n], "seed %d row-major n=%d" % (seed, n))
        assert np.array_equal(out[:, n:], C0[:, n:]), "padding columns of C were touched"
        # column-major: B is k x n with leading dimension ldbc >= k, C is m x n with ldcc >= m
        ldbc, ldcc = a.cols + int(rng.integers(0, 3)), a.rows + int(rng.integers(0, 3))
        Bc = wl.uniform(ldbc * n, dtype, 7).reshape(n, ldbc)
        Cc = wl.uniform(ldcc * n, dtype, 8).reshape(n, ldcc)
        announce("spmm random structure, column-major", seed, a.name, n, ldbc, ldcc)
        outc = run_csrmm(gpu, da, capi.ALPHA_SPARSE_LAYOUT_COLUMN_MAJOR, 0, alpha, Bc, ldbc, beta, Cc, ldcc, n, a.cols)
        check(a, alpha, Bc[:, :a.cols].T, beta, Cc[:, :a.rows].T, outc.reshape(n, ldcc)[:, :a.rows].T,
              "seed %d column-major n=%d" % (seed, n))
        assert np.array_equal(outc.reshape(n, ldcc)[:, a.rows:], Cc[:, a.rows:]), "padding rows of C were touched"
    finally:
        da.free()


@pytest.mark.parametrize("maker", [lambda: wl.stencil3d(64, 60, 56, np.float32), lambda: wl.uniform_rows(215040, 215040, 12, np.float32)],
                         ids=["stencil", "random_columns"])
def test_row_major_operand_of_the_middle_sizes(gpu, maker):
    """A dense operand of 48 to 384 MiB, beyond an XCD's L2 and around the size of the memory-side cache: matrices whose
    neighbouring rows share columns and matrices whose rows do not, twice each, against the oracle."""
    a = maker()
    n = 64
    assert 48 << 20 < a.cols * n * 4 <= 384 << 20
    B = wl.uniform(a.cols * n, np.float32, 5).reshape(a.cols, n)
    C0 = wl.uniform(a.rows * n, np.float32, 6).reshape(a.rows, n)
    da = DeviceCsr(a)
    try:
        for rep in range(2):
            announce("spmm row-major, operand of the middle sizes", a.name, rep)
            C = run_csrmm(gpu, da, capi.ALPHA_SPARSE_LAYOUT_ROW_MAJOR, 0, 1.25, B, n, 0.5, C0, n, n, a.cols)
            check(a, 1.25, B, 0.5, C0, C.reshape(a.rows, n), "%s rep %d" % (a.name, rep))
    finally:
        da.free()


@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
@pytest.mark.parametrize("n", [1, 5, 64, 70])
def test_column_major_and_transposed_b(gpu, n, dtype):
    a = wl.uniform_rows(1500, 1200, 16, dtype)
    da = DeviceCsr(a)
    try:
        ldc = a.rows + 3
        C0 = np.asfortranarray(wl.uniform(ldc * n, dtype, 4).reshape(n, ldc).T)          # (ldc, n) column-major
        # op(B) = B: B is k x n column-major with ldb >= k
        ldb = a.cols + 2
        B = np.asfortranarray(wl.uniform(ldb * n, dtype, 5).reshape(n, ldb).T)            # (ldb, n) column-major
        announce("spmm col-major N/N", n, np.dtype(dtype).name)
        out = run_csrmm(gpu, da, capi.ALPHA_SPARSE_LAYOUT_COLUMN_MAJOR, 0, 1.5, B.T.reshape(-1), ldb, 0.5,
                        C0.T.reshape(-1), ldc, n, a.cols)
        out = out.reshape(n, ldc).T
        check(a, 1.5, B[:a.cols, :], 0.5, C0[:a.rows, :], out[:a.rows, :], "col-major n=%d" % n)
        ref_col = orc.csrmm_plain(a, 1.5, np.asfortranarray(B[:a.cols, :]), 0.5, np.asfortranarray(C0[:a.rows, :]), layout="col")
        e = orc.csrmm_err(a, 1.5, np.asfortranarray(B[:a.cols, :]), 0.5, np.asfortranarray(C0[:a.rows, :]),
                          np.asfortranarray(out[:a.rows, :]), ref_col)
        assert e.full <= TOL[a.dtype]
        assert np.array_equal(out[a.rows:, :], C0[a.rows:, :])
        # op(B) = B^T: B is stored n x k column-major (ldb >= n), i.e. the memory of a row-major k x n matrix
        ldb = n + 1
        Bt = wl.uniform(a.cols * ldb, dtype, 5).reshape(a.cols, ldb)                       # row r of op(B) at Bt[r, :n]
        announce("spmm col-major N/T", n, np.dtype(dtype).name)
        out = run_csrmm(gpu, da, capi.ALPHA_SPARSE_LAYOUT_COLUMN_MAJOR, 1, 1.5, Bt.reshape(-1), ldb, 0.5,
                        C0.T.reshape(-1), ldc, n, a.cols)
        out = out.reshape(n, ldc).T
        check(a, 1.5, Bt[:, :n], 0.5, C0[:a.rows, :], out[:a.rows, :], "col-major transB n=%d" % n)
    finally:
        da.free()


@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
def test_host_pointer_mm(gpu, dtype):
    lib = capi.load()
    p, T = capi.prefix(dtype), capi.scalar_type(dtype)
    a = wl.uniform_rows(1000, 800, 16, dtype)
    A = capi.alphasparse_matrix_t()
    rs, re = np.ascontiguousarray(a.row_ptr[:-1]), np.ascontiguousarray(a.row_ptr[1:])
    assert getattr(lib, "alphasparse_%s_create_csr" % p)(byref(A), 0, a.rows, a.cols, capi.ptr(rs), capi.ptr(re),
                                                         capi.ptr(a.col_ind), capi.ptr(a.values)) == 0
    n = 10
    B = wl.uniform(a.cols * n, dtype, 5).reshape(a.cols, n)
    C0 = wl.uniform(a.rows * n, dtype, 4).reshape(a.rows, n)
    C = C0.copy()
    announce("host api mm row-major")
    st = getattr(lib, "alphasparse_%s_mm" % p)(0, T(1.5), A, capi.alpha_matrix_descr(0, 0, 0), 0, capi.ptr(B), n, n, T(0.5), capi.ptr(C), n)
    assert st == 0
    check(a, 1.5, B, 0.5, C0, C, "alphasparse_mm row-major")
    Bf, Cf0 = np.asfortranarray(B), np.asfortranarray(C0)
    Cf = Cf0.copy(order="F")
    announce("host api mm col-major")
    st = getattr(lib, "alphasparse_%s_mm" % p)(0, T(1.5), A, capi.alpha_matrix_descr(0, 0, 0), 1, capi.ptr(Bf), n, a.cols, T(0.5), capi.ptr(Cf), a.rows)
    assert st == 0
    check(a, 1.5, B, 0.5, C0, np.ascontiguousarray(Cf), "alphasparse_mm col-major")
    assert lib.alphasparse_destroy(A) == 0


@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
@pytest.mark.parametrize("mat", sorted(MATS))
def test_column_major_every_matrix_shape_and_scratch_growth(gpu, mat, dtype):
    """Column-major B and C on ragged / skewed / one-based matrices, with the dense width going up and
    down between calls on one handle (its scratch buffer grows, then is reused for smaller products),
    and beta = 0 over a C full of NaN."""
    for base in (0, 1):
        a = MATS[mat](dtype, base)
        da = DeviceCsr(a)
        try:
            for n in (2, 130, 3, 64, 65):
                ldb, ldc = a.cols + 1, a.rows + 2
                B = np.asfortranarray(wl.uniform(ldb * n, dtype, 5).reshape(n, ldb).T)
                C0 = np.asfortranarray(wl.uniform(ldc * n, dtype, 4).reshape(n, ldc).T)
                for alpha, beta in ((1.5, 0.5), (1.0, 0.0)):
                    Cin = C0 if beta != 0 else np.full_like(C0, np.nan)
                    announce("spmm col-major", mat, n, np.dtype(dtype).name, base, alpha, beta)
                    out = run_csrmm(gpu, da, capi.ALPHA_SPARSE_LAYOUT_COLUMN_MAJOR, 0, alpha, B.T.reshape(-1), ldb, beta,
                                    Cin.T.reshape(-1), ldc, n, a.cols).reshape(n, ldc).T
                    check(a, alpha, B[:a.cols, :], beta, np.zeros_like(C0[:a.rows, :]) if beta == 0 else C0[:a.rows, :],
                          out[:a.rows, :], "col-major %s n=%d" % (mat, n))
                    if beta != 0:
                        assert np.array_equal(out[a.rows:, :], C0[a.rows:, :]), "padding rows of C were touched"
        finally:
            da.free()


@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
def test_kernel_abi_with_and_without_workspace(gpu, dtype):
    """asamd_?_csrmm (no workspace: element-wise gathers of column-major B) and asamd_?_csrmm_ws
    (row-major copy of B in the workspace) agree with the oracle; a workspace that is too small is ignored."""
    lib = capi.load()
    a = wl.powerlaw_rmat(11, 1500, dtype)
    n = 37
    p, T = capi.prefix(dtype), capi.scalar_type(dtype)
    B = np.asfortranarray(wl.uniform(a.cols * n, dtype, 5).reshape(n, a.cols).T)
    C0 = np.asfortranarray(wl.uniform(a.rows * n, dtype, 4).reshape(n, a.rows).T)
    st = capi.asamd_dense_strides(1, a.cols, 1, a.rows)
    need = lib.asamd_csrmm_workspace_bytes(a.dtype.itemsize, a.rows, n, a.cols, byref(st))
    assert need >= a.cols * n * a.dtype.itemsize
    row_major = capi.asamd_dense_strides(n, 1, n, 1)
    assert lib.asamd_csrmm_workspace_bytes(a.dtype.itemsize, a.rows, n, a.cols, byref(row_major)) == 0
    da = DeviceCsr(a)
    dB = hiprt.DeviceArray.from_numpy(B.T.reshape(-1))
    ws = hiprt.DeviceArray((need,), np.uint8)
    try:
        outs = []
        for what, w, wb in (("none", None, 0), ("full", ws.c_ptr(), need), ("too small", ws.c_ptr(), need // 2)):
            announce("csrmm_ws workspace", what, np.dtype(dtype).name)
            dC = hiprt.DeviceArray.from_numpy(C0.T.reshape(-1))
            e = getattr(lib, "asamd_%s_csrmm_ws" % p)(None, a.rows, n, a.cols, a.nnz, T(1.5), da.val.c_ptr(), da.row_ptr.c_ptr(),
                                                     da.col.c_ptr(), 0, dB.c_ptr(), T(0.5), dC.c_ptr(), byref(st), w, wb)
            assert e == 0
            hiprt.synchronize()
            out = dC.to_numpy().reshape(n, a.rows).T
            dC.free()
            check(a, 1.5, B, 0.5, C0, out, "csrmm_ws %s" % what)
            outs.append(out)
        assert np.array_equal(outs[0], outs[2])   # both took the fallback
    finally:
        ws.free()
        dB.free()
        da.free()


def _band(rows, cols, width, dtype, base=0, seed=11):
    """Row r holds `width` consecutive columns starting near r * cols / rows: neighbouring rows share nearly all
    their columns."""
    rng = np.random.default_rng(seed)
    start = np.minimum((np.arange(rows, dtype=np.int64) * cols) // rows, cols - width)
    row_ptr = (np.arange(rows + 1, dtype=np.int64) * width + base).astype(np.int32)
    col = (start[:, None] + np.arange(width)[None, :] + base).astype(np.int32).reshape(-1)
    val = rng.uniform(-1, 1, size=rows * width).astype(dtype)
    return wl.Csr(rows, cols, row_ptr, col, val, base, "band(%d,%d,%d)" % (rows, cols, width))


SHARED = {
    # 27-point stencil: nine runs of three consecutive columns per row
    "stencil27": lambda dt, base: wl.stencil3d(20, 18, 16, dt, base=base),
    "laplace": lambda dt, base: wl.laplace2d(90, 70, dt, base=base),
    "band100": lambda dt, base: _band(3000, 2600, 100, dt, base),
    # rows that the sixteen lane groups of a workgroup share
    "band300": lambda dt, base: _band(700, 900, 300, dt, base),
    # a matrix of hardly more rows than one workgroup takes, and one that ends inside a workgroup
    "band_short": lambda dt, base: _band(19, 40, 7, dt, base),
    "band_tail": lambda dt, base: _band(32 * 5 + 3, 400, 9, dt, base),
}


@pytest.mark.parametrize("dtype", [np.float32, np.float64, np.complex64, np.complex128], ids=["f32", "f64", "c64", "c128"])
@pytest.mark.parametrize("mat", sorted(SHARED))
@pytest.mark.parametrize("n", [33, 64, 100, 128])
@pytest.mark.parametrize("kernel", ["chosen", "lds"])
def test_row_major_rows_that_share_columns(gpu, mat, n, dtype, kernel, monkeypatch):
    """Matrices whose neighbouring rows share columns.  Aligned and padded leading dimensions (rows of B that are whole cache
    lines and rows that are not), both bases, beta zero and not.  "lds": with ALSPARSE_AMD_SPMM_LDS in the environment, which
    once chose a kernel and must change nothing."""
    from helpers_shapes import complex_vector, complexify, real_dtype
    if kernel == "lds":
        monkeypatch.setenv("ALSPARSE_AMD_SPMM_LDS", "1")
    else:
        monkeypatch.delenv("ALSPARSE_AMD_SPMM_LDS", raising=False)
    cx = np.iscomplexobj(np.zeros(1, dtype))
    tol = {4: 1e-4, 8: 1e-12}[np.dtype(real_dtype(dtype) if cx else dtype).itemsize]
    for base in (0, 1):
        a = SHARED[mat](real_dtype(dtype) if cx else dtype, base)
        if cx:
            a = complexify(a, dtype)
        da = DeviceCsr(a)
        try:
            for pad_b, pad_c in ((0, 0), (3, 5)):
                ldb, ldc = n + pad_b, n + pad_c
                if cx:
                    Bfull = complex_vector(a.cols * ldb, dtype, 5).reshape(a.cols, ldb)
                    Cfull = complex_vector(a.rows * ldc, dtype, 4).reshape(a.rows, ldc)
                else:
                    Bfull = wl.uniform(a.cols * ldb, dtype, 5).reshape(a.cols, ldb)
                    Cfull = wl.uniform(a.rows * ldc, dtype, 4).reshape(a.rows, ldc)
                for alpha, beta in ((1.5, 0.5), (1.0, 0.0)):
                    announce("spmm rows sharing columns", mat, n, np.dtype(dtype).name, base, ldb, ldc, alpha, beta)
                    out = run_csrmm(gpu, da, capi.ALPHA_SPARSE_LAYOUT_ROW_MAJOR, 0, alpha, Bfull, ldb, beta, Cfull, ldc, n, a.cols)
                    B2, C02, C2 = (np.ascontiguousarray(v) for v in (Bfull[:, :n], Cfull[:, :n], out[:, :n]))
                    ref = orc.csrmm_plain(a, alpha, B2, beta, C02)
                    err = orc.csrmm_err(a, alpha, B2, beta, C02, C2, ref)
                    assert err.zero_den_mismatch == 0 and err.full <= tol, "%s n=%d: %r" % (mat, n, err)
                    if beta == 0:
                        assert err.strict <= tol, "%s n=%d: %r" % (mat, n, err)
                    assert np.array_equal(out[:, n:], Cfull[:, n:]), "padding columns of C were touched"
                    # the same bits on a second run: a row's parts and their order depend on its entries alone
                    again = run_csrmm(gpu, da, capi.ALPHA_SPARSE_LAYOUT_ROW_MAJOR, 0, alpha, Bfull, ldb, beta, Cfull, ldc, n, a.cols)
                    assert np.array_equal(out.view(np.uint8), again.view(np.uint8))
        finally:
            da.free()


@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
@pytest.mark.parametrize("lengths", [
    # blocks of sixteen entries, the longest row of one lane group and the first that the workgroup shares, rows beyond a
    # whole tile; the mean keeps short rows of B on four lanes each, whose long rows begin beyond 256
    [0, 1, 15, 16, 17, 31, 255, 256, 257, 0, 1025] + [3] * 300,
    # the same on sixteen and sixty-four lanes (long rows beyond 1024 and 4096)
    [0, 1023, 1024, 1025, 2, 17] + [20] * 90,
    [4095, 4096, 4097, 0, 64] + [100] * 12,
    [20] * 130,
], ids=["few", "some", "many", "even"])
def test_widths_around_the_tiles(gpu, lengths, dtype):
    """Dense widths around every form of the row kernels: whole short rows (one to four loads), 4, 8 and 16 column
    lanes, two loads a lane, several chunks; and, column-major, the panels of 256, 128 and fewer bytes."""
    v = 16 // np.dtype(dtype).itemsize
    a = csr_from_lengths(lengths, 5003, dtype, base=1)
    da = DeviceCsr(a)
    try:
        for n in sorted({1, v - 1, v, v + 1, 2 * v + 1, 3 * v + 1, 4 * v, 4 * v + 1, 8 * v + 1, 12 * v + 1, 16 * v - 1, 16 * v,
                         16 * v + 1, 24 * v + 3, 32 * v + 1}):
            if n == 0:
                continue
            B = wl.uniform(a.cols * n, dtype, 7)
            C0 = wl.uniform(a.rows * n, dtype, 8)
            announce("spmm around the tiles", len(lengths), n, np.dtype(dtype).name)
            for beta in (0.0, 0.5):
                out = run_csrmm(gpu, da, capi.ALPHA_SPARSE_LAYOUT_ROW_MAJOR, 0, 1.25, B, n, beta, C0, n, n, a.cols)
                check(a, 1.25, B.reshape(-1, n), beta, C0.reshape(-1, n), out.reshape(-1, n), "row-major n=%d" % n)
                out = run_csrmm(gpu, da, capi.ALPHA_SPARSE_LAYOUT_COLUMN_MAJOR, 0, 1.25, B, a.cols, beta, C0, a.rows, n, a.cols)
                check(a, 1.25, B.reshape(n, -1).T, beta, C0.reshape(n, -1).T, out.reshape(n, -1).T, "column-major n=%d" % n)
    finally:
        da.free()


@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
@pytest.mark.parametrize("n", [1, 5, 70])
def test_kernel_abi_without_entries(gpu, n, dtype):
    """asamd_?_csrmm_ws on a matrix without entries, whose arrays hold nothing: C = beta * C in both layouts.  (The public
    calls return before that and leave C alone.)"""
    lib = capi.load()
    m, k = 100, 30
    T = capi.scalar_type(dtype)
    C0, B = wl.uniform(m * n, dtype, 4), wl.uniform(k * n, dtype, 5)
    rp, empty = hiprt.DeviceArray.from_numpy(np.ones(m + 1, dtype=np.int32)), hiprt.DeviceArray((0,), dtype)
    dB, ws = hiprt.DeviceArray.from_numpy(B), hiprt.DeviceArray((1 << 20,), np.uint8)
    try:
        for st in (capi.asamd_dense_strides(n, 1, n, 1), capi.asamd_dense_strides(1, k, 1, m), capi.asamd_dense_strides(n, 1, 1, m)):
            for beta in (0.0, 0.5):
                announce("csrmm_ws without entries", n, np.dtype(dtype).name, st.b_row_stride, st.c_row_stride, beta)
                dC = hiprt.DeviceArray.from_numpy(np.full_like(C0, np.nan) if beta == 0 else C0)
                assert getattr(lib, "asamd_%s_csrmm_ws" % capi.prefix(dtype))(
                    None, m, n, k, 0, T(1.5), empty.c_ptr(), rp.c_ptr(), empty.c_ptr(), 1, dB.c_ptr(), T(beta), dC.c_ptr(),
                    byref(st), ws.c_ptr(), 1 << 20) == 0
                hiprt.synchronize()
                assert np.array_equal(dC.to_numpy(), (C0 * dtype(beta)).astype(dtype))
                dC.free()
    finally:
        for d in (rp, empty, dB, ws):
            d.free()


@pytest.mark.parametrize("dtype", [np.float32, np.float64, np.complex128], ids=["f32", "f64", "c128"])
@pytest.mark.parametrize("m,chunks", [(1, 1), (5, 3), (511, 1), (513, 1), (2049, 1), (8191, 1), (8193, 1), (130, 5)])
def test_few_rows_of_many_entries(gpu, m, chunks, dtype):
    """Matrices of so few rows that a workgroup takes one, two, ... sixteen of them (sixty-four with column-major C), and rows
    around the lengths from which its groups share a row (64 to 256, by the rows it takes)."""
    from helpers_shapes import complex_vector
    vector = complex_vector if np.dtype(dtype).kind == "c" else wl.uniform
    rng = np.random.default_rng(m)
    lengths = rng.choice([0, 1, 17, 63, 64, 65, 128, 129, 256, 257], size=m, p=[0.1] * 10 if m < 1000 else [0.3, 0.3, 0.3] + [0.1 / 7] * 7)
    lengths[0] = 1025
    row_ptr = np.concatenate([[0], np.cumsum(lengths)])
    col = rng.integers(0, 900, size=int(row_ptr[-1]))
    a = wl.Csr(m, 900, row_ptr.astype(np.int32), col.astype(np.int32), vector(col.size, dtype, 7), 0, "few rows")
    n = 16 * (16 // np.dtype(dtype).itemsize) * chunks + (chunks > 1)
    B, C0 = vector(900 * n, dtype, 5), vector(m * n, dtype, 4)
    da = DeviceCsr(a)
    try:
        for layout, row, b, c in ((capi.ALPHA_SPARSE_LAYOUT_ROW_MAJOR, True, n, n), (capi.ALPHA_SPARSE_LAYOUT_COLUMN_MAJOR, False, 900, m)):
            announce("spmm few rows", m, n, np.dtype(dtype).name, layout)
            out = run_csrmm(gpu, da, layout, 0, 1.25, B, b, 0.5, C0, c, n, 900)
            B2, C02, C2 = (np.ascontiguousarray(v.reshape(-1, n) if row else v.reshape(n, -1).T) for v in (B, C0, out))
            ref = orc.csrmm_plain(a, 1.25, B2, 0.5, C02)
            err = orc.csrmm_err(a, 1.25, B2, 0.5, C02, C2, ref)
            tol = 1e-4 if np.dtype(dtype) == np.float32 else 1e-12
            assert err.zero_den_mismatch == 0 and err.full <= tol, (m, n, err)
    finally:
        da.free()


def _far_matrix(m, cols, per_row, dtype, base):
    """Rows of random columns of at least sixteen entries on average, some without entries and some that a workgroup shares."""
    rng = np.random.default_rng(m + per_row)
    lengths = np.full(m, per_row)
    lengths[::97], lengths[5::1001], lengths[7::1501] = 0, 300, 257
    row_ptr = np.concatenate([[0], np.cumsum(lengths)])
    return wl.Csr(m, cols, (row_ptr + base).astype(np.int32), (rng.integers(0, cols, size=int(row_ptr[-1])) + base).astype(np.int32),
                  None, base, "far rows")


@pytest.mark.parametrize("dtype", [np.float32, np.float64, np.complex64, np.complex128], ids=["f32", "f64", "c64", "c128"])
@pytest.mark.parametrize("m", [8192, 8207])
def test_two_loads_a_lane_one_row_of_b_in_flight(gpu, m, dtype):
    """Chunks of more than 256 bytes over whole tiles of rows of sixteen entries and more: one and several chunks, the last load
    moved back by every number of columns; both matrices end inside and at the end of a workgroup's tile."""
    from helpers_shapes import complex_vector
    vector = complex_vector if np.dtype(dtype).kind == "c" else wl.uniform
    v = 16 // np.dtype(dtype).itemsize
    a = _far_matrix(m, 3001, 20, dtype, 1)
    a.values = vector(a.col_ind.size, dtype, 7)
    da = DeviceCsr(a)
    try:
        for n in (16 * v + 1, 24 * v + v - 1, 32 * v - 1, 64 * v + 1 if m == 8192 else 17 * v):
            ldb = n + (1 if n % (8 * v) == 0 else 0)  # (rows of B that are whole cache lines take one load a lane)
            assert a.nnz >= 16 * m and (ldb * np.dtype(dtype).itemsize) % 128
            B, C0 = vector(a.cols * ldb, dtype, 5).reshape(a.cols, ldb), vector(m * n, dtype, 4)
            announce("spmm two loads a lane", m, n, np.dtype(dtype).name)
            out = run_csrmm(gpu, da, capi.ALPHA_SPARSE_LAYOUT_ROW_MAJOR, 0, 1.25, B, ldb, 0.5, C0, n, n, a.cols)
            B2, C02, C2 = np.ascontiguousarray(B[:, :n]), C0.reshape(m, n), out.reshape(m, n)
            err = orc.csrmm_err(a, 1.25, B2, 0.5, C02, C2, orc.csrmm_plain(a, 1.25, B2, 0.5, C02))
            tol = 1e-4 if np.dtype(dtype).name in ("float32", "complex64") else 1e-12
            assert err.zero_den_mismatch == 0 and err.full <= tol, (m, n, err)
    finally:
        da.free()


@pytest.mark.parametrize("n", [64, 65])
def test_operands_beyond_the_memory_side_cache(gpu, n):
    """B and C of more than 256 MB together under rows of sixteen entries and more: one row of B in flight with one load a lane,
    row-major C past the caches, and column-major C with B laid out in panels (whole tiles of 64 rows) and with B^T."""
    m, k = 32768 + 9, 1050001
    a = _far_matrix(m, k, 18, np.float32, 0)
    a.values = wl.uniform(a.col_ind.size, np.float32, 7)
    assert a.nnz >= 16 * m and (m + k) * n * 4 > 256e6
    B, C0 = wl.uniform(k * n, np.float32, 5), wl.uniform(m * n, np.float32, 4)
    da = DeviceCsr(a)
    ROW, COL = capi.ALPHA_SPARSE_LAYOUT_ROW_MAJOR, capi.ALPHA_SPARSE_LAYOUT_COLUMN_MAJOR
    try:
        for layout, trans, ldb, ldc in ((ROW, 0, n, n), (COL, 0, k, m), (COL, 1, n, m)):
            announce("spmm beyond the memory-side cache", n, layout, trans)
            out = run_csrmm(gpu, da, layout, trans, 1.25, B, ldb, 0.5, C0, ldc, n, k)
            B2 = B.reshape(n, k).T if (layout, trans) == (COL, 0) else B.reshape(k, n)
            C02, C2 = (x.reshape(m, n) if layout == ROW else x.reshape(n, m).T for x in (C0, out))
            check(a, 1.25, B2, 0.5, C02, C2, "layout %d trans %d n=%d" % (layout, trans, n))
    finally:
        da.free()


@pytest.mark.parametrize("dtype", [np.float32, np.float64, np.complex64, np.complex128], ids=["f32", "f64", "c64", "c128"])
@pytest.mark.parametrize("per_row", [3, 20])
def test_column_major_with_room_for_b_alone(gpu, per_row, dtype):
    """A workspace of as many elements as B has: its copy in panels of powers of two, every width up to a full panel and one
    more; a byte less takes the kernel that gathers B in place."""
    from helpers_shapes import complex_vector
    vector = complex_vector if np.dtype(dtype).kind == "c" else wl.uniform
    lib, size, letter = capi.load(), np.dtype(dtype).itemsize, capi.prefix(dtype)
    scalar = capi.scalar_type(dtype)
    m, k = 530, 401
    a = _far_matrix(m, k, per_row, dtype, 1)
    a.values = vector(a.col_ind.size, dtype, 7)
    da = DeviceCsr(a)
    try:
        for n in sorted({2, 3, 7, 64 // size + 1, 128 // size - 1, 128 // size, 128 // size + 1, 256 // size - 1, 256 // size, 256 // size + 3}):
            st = capi.asamd_dense_strides(1, k, 1, m)
            least = lib.asamd_csrmm_least_workspace_bytes(size, n, k, byref(st))
            most = lib.asamd_csrmm_workspace_bytes(size, m, n, k, byref(st))
            assert k * n * size <= least <= k * n * size + 7 * 512
            B, C0 = vector(k * n, dtype, 5), vector(m * n, dtype, 4)
            dB, ws = hiprt.DeviceArray.from_numpy(B), hiprt.DeviceArray((most + least,), np.uint8)
            B2, C02 = np.ascontiguousarray(B.reshape(n, k).T), np.ascontiguousarray(C0.reshape(n, m).T)
            ref = orc.csrmm_plain(a, 1.25, B2, 0.5, C02)
            for room in (min(least, most) - 1, least, most):
                announce("spmm column-major, workspace", n, np.dtype(dtype).name, per_row, room)
                dC = hiprt.DeviceArray.from_numpy(C0)
                assert getattr(lib, "asamd_%s_csrmm_ws" % letter)(
                    None, m, n, k, a.nnz, scalar(1.25), da.val.c_ptr(), da.row_ptr.c_ptr(), da.col.c_ptr(), 1, dB.c_ptr(),
                    scalar(0.5), dC.c_ptr(), byref(st), ws.c_ptr(), room) == 0
                hiprt.synchronize()
                C2 = np.ascontiguousarray(dC.to_numpy().reshape(n, m).T)
                err = orc.csrmm_err(a, 1.25, B2, 0.5, C02, C2, ref)
                tol = 1e-4 if np.dtype(dtype).name in ("float32", "complex64") else 1e-12
                assert err.zero_den_mismatch == 0 and err.full <= tol, (n, room, err)
                dC.free()
            dB.free()
            ws.free()
    finally:
        da.free()
