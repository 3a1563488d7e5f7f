"""Merge-path without a table of coordinates: every workgroup finds its own two, 64 probes at a time.  Compared with the
CPU oracle at one workgroup, at the edges of two and three, and with runs of empty rows and rows longer than workgroups."""
import numpy as np
import pytest

from alsparse_amd import workloads as wl
from helpers import DeviceCsr, announce, check_spmv, run_plan_csrmv
from helpers_shapes import csr_from_lengths

pytestmark = pytest.mark.gpu

LENGTHS = {
    "one workgroup": [3] * 100,
    "edge of two": [1] * 1024,            # rows + entries: exactly two workgroups of 1 024 items, one of 2 048
    "one item more": [1] * 1024 + [0],
    "one item less": [1] * 1023 + [0],
    "65 rows": [0] * 64 + [5000],
    "empty runs": [0] * 3000 + [7000] + [0] * 5000 + [1, 0, 2, 4096, 0] * 3 + [0] * 2000,
    "nothing but a long row": [20000],
    "skewed": [int(30000 / (i + 1)) for i in range(4000)],
}


@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
@pytest.mark.parametrize("base", [0, 1])
@pytest.mark.parametrize("shape", list(LENGTHS))
def test_workgroups_find_their_coordinates(gpu, shape, base, dtype):
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
