"""coomv where a wave's steps of 256 entries (four consecutive ones per lane) can go wrong: row ends at every position in
a lane, runs that cross lanes, steps and waves, a last step that is nearly empty, and arrays off the 16-byte grid."""
from ctypes import byref

import numpy as np
import pytest

from alsparse_amd import capi, hiprt, workloads as wl
from helpers import _ShiftedArray, announce
from helpers_shapes import csr_from_lengths
from oracle import oracle as orc
from test_gpu_formats_mv import check, run_coomv

pytestmark = pytest.mark.gpu


def _lengths(nnz, seed):
    """Row lengths that sum to nnz: mostly 0 .. 9, now and then a run of hundreds."""
    rng = np.random.default_rng(seed)
    out, left = [], nnz
    while left > 0:
        k = int(rng.integers(200, 700)) if rng.random() < 0.01 else int(rng.integers(0, 10))
        out.append(min(k, left))
        left -= out[-1]
    return out


@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
@pytest.mark.parametrize("nnz", [1, 3, 4, 5, 255, 256, 257, 1023, 1024, 1025, 4095, 4097, 20011])
def test_edges_of_steps_and_waves(gpu, dtype, nnz):
    a = csr_from_lengths(_lengths(nnz, nnz), 3000, dtype, seed=nnz)
    x, y0 = wl.uniform(a.cols, dtype, 3), wl.uniform(a.rows, dtype, 4)
    rows = orc.csr2coo(a)
    for base, alpha, beta in ((0, 1.0, 0.0), (1, -1.5, 0.5)):
        announce("coomv steps", np.dtype(dtype).name, "nnz", nnz, "base", base)
        y = run_coomv(gpu, a.rows, a.cols, a.values, rows + base, a.col_ind + base, base, alpha, x, beta, y0)
        check(a, alpha, x, beta, y0, y, orc.coomv_plain(a, rows, alpha, x, beta, y0), "nnz %d" % nnz)


@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
@pytest.mark.parametrize("shift", [1, 2, 3])
def test_arrays_off_the_128_bit_grid(gpu, dtype, shift):
    a = csr_from_lengths(_lengths(5003, shift), 3000, dtype, seed=shift)
    x, y0 = wl.uniform(a.cols, dtype, 3), wl.uniform(a.rows, dtype, 4)
    rows = orc.csr2coo(a)
    lib, T, d = capi.load(), capi.scalar_type(dtype), capi.make_descr(base=0)
    arrays = [_ShiftedArray(v, shift) for v in (a.values, rows.astype(np.int32), a.col_ind)]
    dx, dy = hiprt.DeviceArray.from_numpy(x), hiprt.DeviceArray.from_numpy(y0)
    al, be = T(1.5), T(0.5)
    announce("coomv shifted arrays", np.dtype(dtype).name, "by", shift)
    try:
        assert getattr(lib, "alphasparse_dcu_%s_coomv" % capi.prefix(np.dtype(dtype)))(
            gpu.h, 0, a.rows, a.cols, a.nnz, byref(al), byref(d), arrays[0].c_ptr(), arrays[1].c_ptr(), arrays[2].c_ptr(),
            dx.c_ptr(), byref(be), dy.c_ptr()) == 0
        hiprt.synchronize()
        check(a, 1.5, x, 0.5, y0, dy.to_numpy(), orc.coomv_plain(a, rows, 1.5, x, 0.5, y0), "shift %d" % shift)
    finally:
        for v in arrays + [dx, dy]:
            v.free()
