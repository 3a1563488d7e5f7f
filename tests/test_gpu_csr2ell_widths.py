"""csr2ell at the widths where a workgroup's rows change (256, 128, 64, 32, and more than 32 rows fit): bit-exact against
the oracle, a last workgroup that ends inside the matrix, arrays on and off the 16-byte grid."""
import numpy as np
import pytest

from helpers import DeviceCsr, announce
from helpers_shapes import csr_from_lengths
from oracle import oracle as orc
from test_gpu_convert import gpu_csr2ell

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
@pytest.mark.parametrize("width", [1, 15, 16, 17, 32, 33, 64, 65, 127, 128, 129])
def test_widths_at_which_the_rows_of_a_workgroup_change(gpu, width, dtype):
    rng = np.random.default_rng(width)
    lengths = np.where(rng.random(701) < 0.7, width, rng.integers(0, width + 1, size=701))
    lengths[5] = width
    for shift in (0, 1):
        a = csr_from_lengths(lengths, 4000, dtype, seed=width, base=shift)
        da = DeviceCsr(a, shift)
        try:
            announce("csr2ell width", width, np.dtype(dtype).name, "shift", shift)
            w, ev, ec = gpu_csr2ell(gpu, da, 1 - shift)
            assert w == orc.csr2ell_width(a) == width
            rv, rc = orc.csr2ell(a, ell_base=1 - shift)
            assert np.array_equal(ev.view(np.uint8), rv.view(np.uint8)) and np.array_equal(ec, rc)
        finally:
            da.free()
