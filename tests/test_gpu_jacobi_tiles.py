"""FP32 Jacobi passes of two and three sweeps on tiles: the bits of the one-column strips at the edges of the
tiles (28 x 12 x 6 and 26 x 10 x 6 stored points), on thin grids and for every remainder of the sweep count."""
import ctypes

import numpy
import pytest

pytestmark = pytest.mark.gpu


def _sweeps(shape, rho, v0, sweeps, block):
    import torch
    from qmtools import _native as nat
    g = nat.geom((*shape, 0.3, (0.0, 0.0, 0.0)))
    dr, dv = torch.tensor(rho, device="cuda"), torch.tensor(v0, device="cuda")
    done, delta = ctypes.c_int64(0), ctypes.c_double(0)
    nat.call("qm_jacobi", nat.stream(), ctypes.byref(g), nat.QM_PREC_FP32, nat.dptr(dr), nat.dptr(dv), None, sweeps,
             -1.0, block, ctypes.byref(done), ctypes.byref(delta))
    assert done.value == sweeps
    dt = torch.tensor(v0, device="cuda")
    vp = ctypes.c_void_p
    nat.call("qm_jacobi_batch", nat.stream(), 1, ctypes.byref(g), (vp * 1)(dr.data_ptr()), (vp * 1)(dt.data_ptr()),
             (vp * 1)(0), nat.QM_PREC_FP32, sweeps, block, 1)
    return dv.cpu().numpy(), dt.cpu().numpy()


@pytest.mark.parametrize("shape", [(3, 3, 3), (1, 5, 4), (26, 10, 6), (28, 12, 6), (29, 13, 7), (57, 25, 13),
                                   (5, 61, 33), (150, 150, 141)])
def test_tiles_give_the_bits_of_strips(shape):
    from qmtools import autotune
    n = shape[0] * shape[1] * shape[2]
    rng = numpy.random.default_rng(4)
    rho, v0 = rng.standard_normal(n), rng.standard_normal(n)
    old = autotune.get("jacobi_pairs")
    try:
        for sweeps, block in ((1, 2), (2, 2), (9, 4), (17, 6), (23, 8), (64, 50)):
            out = []
            for knob in (1, 0):
                autotune.set("jacobi_pairs", knob)
                print("[case] jacobi tiles", shape, sweeps, block, knob, flush=True)
                out += _sweeps(shape, rho, v0, sweeps, block)
            for other in out[1:]:
                numpy.testing.assert_array_equal(other, out[0])
    finally:
        autotune.set("jacobi_pairs", old)
