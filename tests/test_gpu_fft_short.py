"""FFT Poisson solve on axes of up to 10 points (transforms of 2 to 20)."""
import ctypes

import numpy
import pytest
from conftest import BASIS
from test_gpu_fft_real import _periodic

pytestmark = pytest.mark.gpu


def _call(shape, q, prec, mode):
    import torch
    import qmtools as qm
    from qmtools import _native as nat, synth
    from qmtools.qmtools import device_molecule
    mol = synth.synthetic_molecule(5, 3, qm.BasisSet(BASIS))
    h = 0.3
    o = mol.coords.mean(axis=0) - 0.5 * numpy.array(shape) * h
    dq = torch.tensor(q, device="cuda")
    v = torch.full_like(dq, float("nan"))
    g = nat.geom((*shape, h, tuple(o)))
    dm = device_molecule(mol)

    def run():
        nat.call("qm_hartree_fft", dm.handle, nat.stream(), ctypes.byref(g), prec, nat.QM_F64, nat.dptr(dq), 0.2, 6.0,
                 mode, nat.dptr(v))
    return mol, h, o, v, run


@pytest.mark.parametrize("shape", [(2, 4, 6), (4, 6, 8), (6, 8, 10), (8, 10, 4), (10, 4, 2), (8, 8, 8), (3, 4, 5),
                                   (5, 3, 4), (4, 5, 3), (9, 2, 7)])
def test_short_axes(shape):
    """The gates of the FFT solve: 1e-10 in FP64 and 1e-6 in complex64 of the largest value."""
    from oracle import fft as off
    from qmtools import _native as nat
    q = numpy.random.default_rng(3).uniform(0.0, 0.01, shape).ravel()
    for mode in ("periodic", "freespace"):
        cmode = {"periodic": nat.QM_FFT_PERIODIC, "freespace": nat.QM_FFT_FREESPACE}[mode]
        for prec, tol in ((nat.QM_PREC_FP64, 1e-10), (nat.QM_PREC_FP32, 1e-6)):
            print("[case] fft short axes", shape, mode, prec, flush=True)
            mol, h, o, v, run = _call(shape, q, prec, cmode)
            args = (q, mol.types, mol.coords, *shape, h, o)
            want = (_periodic(off.total_charge_rhs(*args), h / off.ANG2BOR) if mode == "periodic"
                    else off.hartree_fft(*args, mode=mode))
            run()
            got = v.cpu().numpy().reshape(shape)
            assert numpy.abs(got - want).max() <= tol * numpy.abs(want).max(), (mode, prec)


def test_eight_points_cost_no_more_than_sixteen():
    """8^3 periodic points take at most 1.5 times as long as 16^3."""
    import torch
    from qmtools import _native as nat

    def best(n):
        run = _call((n, n, n), numpy.full(n ** 3, 0.01), nat.QM_PREC_FP64, nat.QM_FFT_PERIODIC)[4]
        t = 1e9
        for _ in range(8):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            for _ in range(4):
                run()
            b.record()
            b.synchronize()
            t = min(t, a.elapsed_time(b))
        return t
    print("[case] fft short axes, time", flush=True)
    assert best(8) <= 1.5 * best(16)


@pytest.mark.parametrize("n,prec,ok", [(2560, "FP64", True), (2558, "FP64", True), (2561, "FP64", False),
                                       (2564, "FP64", False), (2638, "FP64", False), (3840, "FP64", True),
                                       (3888, "FP64", False), (3969, "FP64", False), (4096, "FP64", False),
                                       (2564, "FP32", True), (3969, "FP32", True), (4096, "FP32", True)])
def test_length_limits(n, prec, ok):
    """Lengths beyond the documented limits are refused, whatever the axis."""
    from qmtools import _native as nat
    for axis in range(3):
        shape = [2, 2, 2]
        shape[axis] = n
        print("[case] fft length", shape, prec, flush=True)
        run = _call(tuple(shape), numpy.full(4 * n, 0.01), getattr(nat, "QM_PREC_" + prec), nat.QM_FFT_PERIODIC)[4]
        if ok:
            run()
        else:
            with pytest.raises(nat.QMError) as e:
                run()
            assert e.value.code == nat.QM_ELIMIT
