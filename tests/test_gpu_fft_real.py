"""FFT Poisson solve on half spectra: odd counts of lines, odd, prime and single-stage lengths on each axis."""
import math

import numpy
import pytest
from conftest import BASIS

pytestmark = pytest.mark.gpu


def _periodic(rhs, h_ang):
    """Full complex transforms with the solver's frequencies: index i counts as i below n // 2, else i - n
    (kernel_fft.cu:82-106; for odd n that is not the symmetric choice)."""
    k2 = 0.0
    for axis, n in enumerate(rhs.shape):
        i = numpy.arange(n)
        k = numpy.where(i > n // 2 - 1, i - n, i) / (n * h_ang)
        k2 = k2 + (k ** 2).reshape([-1 if a == axis else 1 for a in range(3)])
    k2[0, 0, 0] = 1.0
    f = -1.0 / (4.0 * math.pi ** 2 * k2)
    f[0, 0, 0] = 0.0
    return numpy.fft.ifftn(numpy.fft.fftn(rhs) * f).real


@pytest.mark.parametrize("shape", [(2, 3, 2), (3, 2, 5), (7, 10, 9), (11, 13, 16), (35, 16, 33), (16, 35, 30),
                                   (100, 9, 14), (12, 36, 257), (64, 65, 20)])
def test_half_spectrum_lengths(shape):
    """The gates of the FFT solve: 1e-10 in FP64 and 1e-6 in complex64 of the largest value."""
    import ctypes
    import torch
    import qmtools as qm
    from oracle import fft as off
    from qmtools import _native as nat, synth
    from qmtools.qmtools import device_molecule
    mol = synth.synthetic_molecule(5, 3, qm.BasisSet(BASIS))
    h = 0.3
    o = mol.coords.mean(axis=0) - 0.5 * numpy.array(shape) * h
    q = numpy.random.default_rng(3).uniform(0.0, 0.01, shape).ravel()
    args = (q, mol.types, mol.coords, *shape, h, o)
    dq = torch.tensor(q, device="cuda")
    for mode in ("periodic", "freespace"):
        if mode == "periodic":
            want = _periodic(off.total_charge_rhs(*args), h / off.ANG2BOR)
        else:
            want = off.hartree_fft(*args, mode=mode)
        cmode = {"periodic": nat.QM_FFT_PERIODIC, "freespace": nat.QM_FFT_FREESPACE}[mode]
        for prec, tol in ((nat.QM_PREC_FP64, 1e-10), (nat.QM_PREC_FP32, 1e-6)):
            print("[case] fft half spectrum", shape, mode, prec, flush=True)
            v = torch.full_like(dq, float("nan"))
            nat.call("qm_hartree_fft", device_molecule(mol).handle, nat.stream(),
                     ctypes.byref(nat.geom((*shape, h, tuple(o)))), prec, nat.QM_F64, nat.dptr(dq), 0.2, 6.0, cmode,
                     nat.dptr(v))
            got = v.cpu().numpy().reshape(shape)
            assert numpy.abs(got - want).max() <= tol * numpy.abs(want).max(), (mode, prec)
