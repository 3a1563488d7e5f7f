"""The work that users of this library have it do, as timed cases through the public C API.

A case is a plain dict: an operation (csrmv, csrmm, coomv, ellmv, or the conversions), a matrix family with its sizes, an
element type and the call's options.  ``listed()`` holds a fixed choice, ``draw()`` gives more of the same ranges,
``prepare()`` makes what a program has in hand before the call (device arrays, handle, the analysis where the program
makes one) and ``run()`` is the call itself.

Matrix families:

* ``points``     random (row, column) positions, duplicates merged: a small unstructured matrix
* ``laplace2d``  5-point Laplacian on nx x ny points, diagonal 4, neighbours -1 (random coefficients for the conversions)
* ``stencil3d``  27-point stencil on nx x ny x nz points: a trilinear finite-element matrix
* ``uniform``    ``per_row`` distinct sorted uniform columns in every row
* ``powerlaw``   Zipf(2) row lengths, R-MAT columns: a graph
"""
import math
from ctypes import byref, c_int32, c_void_p

import numpy as np
import torch

from alsparse_amd import capi

#: per element type: torch type of the values, real torch type, the C API's letter, bytes, numpy type
TYPES = {
    "f32": (torch.float32, torch.float32, "s", 4, np.float32),
    "f64": (torch.float64, torch.float64, "d", 8, np.float64),
    "c64": (torch.complex64, torch.float32, "c", 8, np.complex64),
    "c128": (torch.complex128, torch.float64, "z", 16, np.complex128),
}

#: a drawn case moves at most what the largest listed one does (the 16 M-row matrix)
MOST_BYTES = 2.42e9


def listed():
    return [
        # The smallest calls: a 1000 x 1000 matrix with 5000 random points, no analysis, as the reference's test programs
        # call csrmv (info = NULL), one product with A and one with its transpose as in a step of BiCG.  Launches and the
        # host path are all of it.
        {"name": "csrmv_points_1k_pair_f32", "op": "csrmv", "family": "points", "rows": 1000, "cols": 1000, "points": 5000,
         "dtype": "f32", "analysed": False, "trans": "both", "alpha": 1.0, "beta": 0.0},
        # A small graph in double precision, not analysed either: an iterative method that updates a vector in place.
        {"name": "csrmv_powerlaw_50k_f64", "op": "csrmv", "family": "powerlaw", "rows": 50021, "max_len": 20000,
         "dtype": "f64", "analysed": False, "trans": "no", "alpha": 1.0, "beta": 0.5},
        # The matrix of a Poisson solver: two-dimensional 5-point Laplacian, double precision, analysed once.
        {"name": "csrmv_laplace2d_4m_f64", "op": "csrmv", "family": "laplace2d", "nx": 2048, "ny": 2048,
         "dtype": "f64", "analysed": True, "trans": "no", "alpha": 1.0, "beta": 0.0},
        # The largest: 16 entries in each of 16 M rows, columns all over the matrix.
        {"name": "csrmv_uniform_16m_f32", "op": "csrmv", "family": "uniform", "rows": 16777216, "cols": 16777216, "per_row": 16,
         "dtype": "f32", "analysed": True, "trans": "no", "alpha": 1.0, "beta": 0.5},
        # A large graph (page rank, label propagation): very uneven rows, columns that crowd into hubs.
        {"name": "csrmv_powerlaw_8m_f32", "op": "csrmv", "family": "powerlaw", "rows": 8388608, "max_len": 200000,
         "dtype": "f32", "analysed": True, "trans": "no", "alpha": 1.0, "beta": 0.0},
        # A Helmholtz-like operator: 27-point stencil with complex values, on a grid whose sizes are no powers of two.
        {"name": "csrmv_stencil3d_1m_c64", "op": "csrmv", "family": "stencil3d", "nx": 101, "ny": 100, "nz": 97,
         "dtype": "c64", "analysed": True, "trans": "no", "alpha": 1.0, "beta": 0.0},
        # The transposed product of a rectangular matrix (least squares), analysed for it.
        {"name": "csrmv_trans_uniform_1m_f64", "op": "csrmv", "family": "uniform", "rows": 1000003, "cols": 786433, "per_row": 16,
         "dtype": "f64", "analysed": True, "trans": "yes", "alpha": 1.0, "beta": 0.0},
        # Sparse times dense, row-major, 64 columns, columns of A at random (graph features).
        {"name": "csrmm_uniform_1m_n64_f32", "op": "csrmm", "family": "uniform", "rows": 1048576, "cols": 1048576, "per_row": 32,
         "n": 64, "layout": "row", "dtype": "f32", "alpha": 1.5, "beta": 0.5},
        # Sparse times dense, row-major, 64 columns, a finite-element matrix (block Krylov methods).
        {"name": "csrmm_stencil3d_1m_n64_f32", "op": "csrmm", "family": "stencil3d", "nx": 128, "ny": 128, "nz": 64,
         "n": 64, "layout": "row", "dtype": "f32", "alpha": 1.0, "beta": 0.0},
        # The reference's own csrmm layout, column-major, double precision, a ragged number of columns.
        {"name": "csrmm_col_uniform_262k_n17_f64", "op": "csrmm", "family": "uniform", "rows": 262147, "cols": 262147, "per_row": 16,
         "n": 17, "layout": "col", "dtype": "f64", "alpha": 1.0, "beta": 0.0},
        # SpMV on the coordinate form that csr2coo makes.
        {"name": "coomv_laplace2d_6m_f32", "op": "coomv", "family": "laplace2d", "nx": 3001, "ny": 2003,
         "dtype": "f32", "alpha": 1.0, "beta": 0.0},
        # Both conversions of a CSR matrix (a Laplacian with variable coefficients): to COO, and to ELL with the width
        # found first.
        {"name": "convert_laplace2d_4m_f64", "op": "convert", "family": "laplace2d", "nx": 2048, "ny": 2048, "dtype": "f64"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_family(rng, family, most_rows):
    if family == "points":
        rows = _log_int(rng, 300, 60000)
        return {"rows": rows, "cols": _log_int(rng, 300, 60000), "points": rows * rng.randint(2, 12)}
    if family == "laplace2d":
        rows = _log_int(rng, 4000, most_rows)
        nx = max(20, int(math.sqrt(rows) * math.exp(rng.uniform(-0.7, 0.7))))
        return {"nx": nx, "ny": max(20, rows // nx)}
    if family == "stencil3d":
        side = (_log_int(rng, 8000, min(most_rows, 4200000))) ** (1 / 3)
        return {k: max(12, int(side * math.exp(rng.uniform(-0.3, 0.3)))) for k in ("nx", "ny", "nz")}
    if family == "uniform":
        rows = _log_int(rng, 2000, most_rows)
        cols = rows if rng.random() < 0.6 else _log_int(rng, max(2000, rows // 8), min(most_rows, rows * 4))
        return {"rows": rows, "cols": cols, "per_row": _log_int(rng, 3, 64)}
    return {"rows": _log_int(rng, 5000, min(most_rows, 8388608)), "max_len": 0}


def draw(rng):
    """One more case of the ranges the listed ones stand for."""
    while True:
        op = rng.choice(("csrmv",) * 6 + ("csrmm",) * 3 + ("coomv", "ellmv", "convert"))
        dtype = rng.choice(("f32", "f32", "f32", "f64", "f64", "c64", "c128"))
        c = {"op": op, "dtype": dtype}
        if op == "csrmv":
            c["family"] = rng.choice(("points", "laplace2d", "stencil3d", "uniform", "uniform", "powerlaw"))
            # programs that make no analysis have small matrices
            c["analysed"] = rng.random() < 0.7
            c.update(_draw_family(rng, c["family"], 16777216 if c["analysed"] else 400000))
            c["trans"] = "yes" if c["analysed"] and rng.random() < 0.2 else "no"
        elif op == "csrmm":
            c["family"] = rng.choice(("laplace2d", "stencil3d", "uniform", "uniform", "powerlaw"))
            c.update(_draw_family(rng, c["family"], 2097152))
            c["n"] = _log_int(rng, 2, 256)
            c["layout"] = rng.choice(("row", "row", "col"))
        else:
            c["family"] = rng.choice(("laplace2d", "stencil3d", "uniform"))
            c.update(_draw_family(rng, c["family"], 8388608))
        if c["family"] == "powerlaw":
            c["max_len"] = max(100, c["rows"] // 40)
        if op != "convert":
            c["alpha"] = rng.choice((1.0, 1.0, 1.5))
            c["beta"] = rng.choice((0.0, 0.0, 0.5))
        size = work(c)["bytes"]
        if op == "csrmv" and size < 16e6:
            c["trans"] = "both"  # one launch of a small kernel measures little but the launch: small systems take the pair
        elif op != "csrmv" and size < 16e6:
            continue
        if size <= MOST_BYTES and _entries(c) <= 1 << 28:
            return c


# ---- the matrices -----------------------------------------------------------------------------------------------
def _shape(case):
    f = case["family"]
    if f == "laplace2d":
        return (case["nx"] * case["ny"],) * 2
    if f == "stencil3d":
        return (case["nx"] * case["ny"] * case["nz"],) * 2
    return (case["rows"], case["rows"] if f == "powerlaw" else case["cols"])


def _entries(case):
    """Entries of the matrix; for the random families whose duplicates merge, about."""
    f = case["family"]
    if f == "points":
        return case["points"]
    if f == "laplace2d":
        return 5 * case["nx"] * case["ny"] - 2 * (case["nx"] + case["ny"])
    if f == "stencil3d":
        return (3 * case["nx"] - 2) * (3 * case["ny"] - 2) * (3 * case["nz"] - 2)
    if f == "uniform":
        return case["rows"] * min(case["per_row"], case["cols"])
    # Zipf(2) clipped: about ln(max) + 1/2 draws a row, less the repeats that merge
    return int(case["rows"] * (math.log(case["max_len"]) + 0.5) * 0.9)


def _row_ptr(counts):
    row_ptr = torch.zeros(counts.numel() + 1, dtype=torch.int32, device="cuda")
    row_ptr[1:] = torch.cumsum(counts, 0)
    return row_ptr


def _structure(case, gen):
    """row_ptr, col_ind (zero-based, columns ascending) on the GPU."""
    f = case["family"]
    rows, cols = _shape(case)
    if f == "uniform":
        k = min(case["per_row"], cols)
        # a sorted draw from [0, cols - k] plus 0, 1, 2, ... is a sorted draw without repeats
        col = torch.randint(0, cols - k + 1, (rows, k), generator=gen, dtype=torch.int32, device="cuda")
        col = torch.sort(col, dim=1)[0]
        col += torch.arange(k, dtype=torch.int32, device="cuda")
        return torch.arange(rows + 1, dtype=torch.int32, device="cuda") * k, col.reshape(-1)
    if f in ("points", "powerlaw"):
        if f == "points":
            row = torch.randint(0, rows, (case["points"],), generator=gen, device="cuda")
            col = torch.randint(0, cols, (case["points"],), generator=gen, device="cuda")
        else:
            u = 1.0 - torch.rand(rows, generator=gen, dtype=torch.float64, device="cuda")
            length = torch.clamp(torch.floor(1.0 / u), max=case["max_len"]).to(torch.int64)
            row = torch.repeat_interleave(torch.arange(rows, device="cuda"), length)
            levels = max(1, (rows - 1).bit_length())
            col = torch.zeros_like(row)
            for bit in range(levels - 1, -1, -1):  # R-MAT quadrants 0.57, 0.19 / 0.19, 0.05, the row given
                one = torch.where(((row >> bit) & 1).bool(), 5.0 / 24.0, 0.25)
                col = 2 * col + (torch.rand(row.numel(), generator=gen, device="cuda") < one)
            col %= cols
        key = torch.unique_consecutive(torch.sort(row * cols + col)[0])
        row = key // cols
        return _row_ptr(torch.bincount(row, minlength=rows)), (key - row * cols).to(torch.int32)
    # grids, x fastest: the neighbours that exist, columns ascending
    idx = torch.arange(rows, dtype=torch.int32, device="cuda")
    nx, ny, nz = case["nx"], case["ny"], case.get("nz", 1)
    ix, iy, iz = idx % nx, (idx // nx) % ny, idx // (nx * ny)
    if f == "laplace2d":
        steps = ((0, -1, 0), (0, 0, -1), (0, 0, 0), (0, 0, 1), (0, 1, 0))
    else:
        steps = [(dz, dy, dx) for dz in (-1, 0, 1) for dy in (-1, 0, 1) for dx in (-1, 0, 1)]

    def exists(dz, dy, dx):
        return ((ix + dx >= 0) & (ix + dx < nx) & (iy + dy >= 0) & (iy + dy < ny) & (iz + dz >= 0) & (iz + dz < nz))

    there = torch.stack([exists(*s) for s in steps], dim=1)
    col = torch.stack([idx + ((dz * ny + dy) * nx + dx) for dz, dy, dx in steps], dim=1)
    return _row_ptr(there.sum(1)), col[there]


def _uniform(n, case, gen, lo=-1.0, hi=1.0):
    vt, rt = TYPES[case["dtype"]][:2]
    if vt.is_complex:
        return torch.view_as_complex(torch.rand((n, 2), generator=gen, dtype=rt, device="cuda") * (hi - lo) + lo)
    return torch.rand(n, generator=gen, dtype=rt, device="cuda") * (hi - lo) + lo


def _values(case, gen, row_ptr, col):
    vt = TYPES[case["dtype"]][0]
    if case["family"] == "laplace2d" and case["op"] != "convert":
        rows = _shape(case)[0]
        row = torch.repeat_interleave(torch.arange(rows, dtype=torch.int32, device="cuda"),
                                      (row_ptr[1:] - row_ptr[:-1]).to(torch.int64))
        return torch.where(row == col, 4.0, -1.0).to(vt)
    return _uniform(col.numel(), case, gen, 0.0 if case["family"] == "powerlaw" else -1.0)


# ---- what a program holds ---------------------------------------------------------------------------------------
_handle = None


def _the_handle():
    """One library handle for the program, on the default stream (torch's too)."""
    global _handle
    if _handle is None:
        _handle = capi.Handle()
    return _handle.h


def _p(t):
    return c_void_p(t.data_ptr())


def _ok(status):
    if status != capi.ALPHA_SPARSE_STATUS_SUCCESS:
        raise RuntimeError("the library returned status %d" % status)


class State:
    """Device arrays, the argument lists of the calls, and the analysis."""

    def __init__(self):
        self.info = None
        self.calls = []  # (function, arguments)
        self.out = None
        self.keep = []

    def __del__(self):
        if self.info is not None:
            capi.load().alphasparse_dcu_destroy_mat_info(self.info)
            self.info = None


def prepare(case, seed):
    lib, h, s = capi.load(), _the_handle(), State()
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed))
    vt, _, letter, _, npt = TYPES[case["dtype"]]
    T = capi.scalar_type(npt)
    m, n = _shape(case)
    row_ptr, col = _structure(case, gen)
    val = _values(case, gen, row_ptr, col)
    nnz = col.numel()
    descr = capi.make_descr()
    alpha, beta = T(case.get("alpha", 1.0)), T(case.get("beta", 0.0))
    s.keep = [row_ptr, col, val, descr, alpha, beta]
    d = byref(descr)
    op = case["op"]

    def api(name):
        return getattr(lib, name.format(s=letter))

    if op == "csrmv":
        if case["analysed"]:
            t = capi.ALPHA_SPARSE_OPERATION_NON_TRANSPOSE if case["trans"] == "no" else capi.ALPHA_SPARSE_OPERATION_TRANSPOSE
            s.info = capi.alphasparse_dcu_mat_info_t()
            _ok(lib.alphasparse_dcu_create_mat_info(byref(s.info)))
            _ok(api("alphasparse_dcu_{s}_csrmv_analysis")(h, t, m, n, nnz, d, _p(val), _p(row_ptr), _p(col), s.info))
        s.out = []
        for t in {"no": (0,), "yes": (1,), "both": (0, 1)}[case["trans"]]:  # the operation's value in the C API
            x, y = _uniform(m if t else n, case, gen), _uniform(n if t else m, case, gen)
            s.calls.append((api("alphasparse_dcu_{s}_csrmv"),
                            (h, t, m, n, nnz, byref(alpha), d, _p(val), _p(row_ptr), _p(col), s.info, _p(x), byref(beta), _p(y))))
            s.keep += [x, y]
            s.out.append(y)
    elif op == "csrmm":
        w = case["n"]
        row_major = case["layout"] == "row"
        B = _uniform(n * w, case, gen).reshape((n, w) if row_major else (w, n))
        C = _uniform(m * w, case, gen).reshape((m, w) if row_major else (w, m))
        layout = capi.ALPHA_SPARSE_LAYOUT_ROW_MAJOR if row_major else capi.ALPHA_SPARSE_LAYOUT_COLUMN_MAJOR
        s.calls = [(api("alphasparse_dcu_{s}_csrmm"),
                    (h, 0, 0, layout, m, w, n, nnz, byref(alpha), d, _p(val), _p(row_ptr), _p(col), _p(B), B.shape[1],
                     byref(beta), _p(C), C.shape[1]))]
        s.keep += [B, C]
        s.out = C
    else:
        width = c_int32(0)
        wcall = (lib.alphasparse_dcu_csr2ell_width, (h, m, d, _p(row_ptr), d, byref(width)))
        _ok(wcall[0](*wcall[1]))
        coo_row = torch.empty(nnz, dtype=torch.int32, device="cuda")
        coo = (lib.alphasparse_dcu_csr2coo, (h, _p(row_ptr), nnz, m, _p(coo_row), 0))
        ell = None
        if op != "coomv":
            ev = torch.empty((width.value, m), dtype=vt, device="cuda")
            ec = torch.empty((width.value, m), dtype=torch.int32, device="cuda")
            ell = (api("alphasparse_dcu_{s}csr2ell"), (h, m, d, _p(val), _p(row_ptr), _p(col), d, width.value, _p(ev), _p(ec)))
            s.keep += [ev, ec]
        s.keep += [coo_row, width]
        if op == "convert":
            s.calls = [coo, wcall, ell]
            s.out = [coo_row, ev, ec]
            return s
        x, y = _uniform(n, case, gen), _uniform(m, case, gen)
        s.keep += [x, y]
        s.out = y
        if op == "coomv":
            _ok(coo[0](*coo[1]))
            s.calls = [(api("alphasparse_dcu_{s}_coomv"),
                        (h, 0, m, n, nnz, byref(alpha), d, _p(val), _p(coo_row), _p(col), _p(x), byref(beta), _p(y)))]
        else:
            _ok(ell[0](*ell[1]))
            s.calls = [(api("alphasparse_dcu_{s}_ellmv"),
                        (h, 0, m, n, byref(alpha), d, _p(ev), _p(ec), width.value, _p(x), byref(beta), _p(y)))]
    return s


def run(state):
    for fn, args in state.calls:
        status = fn(*args)
        if status:
            _ok(status)
    return state.out


def work(case):
    """Every operand read once, every result written once."""
    size = TYPES[case["dtype"]][3]
    m, n = _shape(case)
    nnz = _entries(case)
    op = case["op"]
    flop = 2 if size in (4, 8) and case["dtype"][0] == "f" else 8
    twice = 2 if case.get("beta", 0.0) != 0.0 else 1
    if op == "csrmm":
        w = case["n"]
        return {"bytes": nnz * (size + 4) + 4 * (m + 1) + n * w * size + m * w * size * twice, "flops": flop * nnz * w}
    if op == "convert":
        slots = m * _width(case)
        return {"bytes": 4 * (m + 1) + 4 * nnz + nnz * (size + 4) + slots * (size + 4), "flops": 0}
    index = {"csrmv": 4 * nnz + 4 * (m + 1), "coomv": 8 * nnz, "ellmv": 0}[op]
    if op == "ellmv":
        matrix = m * _width(case) * (size + 4)
    else:
        matrix = nnz * size + index
    total = 0
    for into, out in {"no": [(n, m)], "yes": [(m, n)], "both": [(n, m), (m, n)]}[case.get("trans", "no")]:
        total += matrix + into * size + out * size * twice
    return {"bytes": total, "flops": flop * nnz * (2 if case.get("trans") == "both" else 1)}


def _width(case):
    return {"laplace2d": 5, "stencil3d": 27}.get(case["family"]) or min(case["per_row"], case["cols"])


def tolerance(case):
    """Sums in another order differ by a few roundings of the element type; conversions only move values."""
    if case["op"] == "convert":
        return "exact"
    return {"rel": 1e-5} if case["dtype"] in ("f32", "c64") else {"rel": 1e-13}
