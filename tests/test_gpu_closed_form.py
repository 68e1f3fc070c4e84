"""Relaxations in closed form by sine transforms: sizes at the edges of the matrix tiles, the convergence
check, and the inputs that are left to the sweeps."""
import ctypes

import numpy
import pytest

pytestmark = pytest.mark.gpu


def _jacobi(shape, rho, v0, sweeps, tol=-1.0, every=0, h=0.3):
    import torch
    from qmtools import _native as nat
    g = nat.geom((*shape, h, (0.0, 0.0, 0.0)))
    dr, dv = torch.tensor(rho, device="cuda"), torch.tensor(v0, device="cuda")
    dt = torch.full_like(dv, 7.0)
    done, delta = ctypes.c_int64(0), ctypes.c_double(0)
    rc = nat.library().qm_jacobi(nat.context(), nat.stream(), ctypes.byref(g), nat.QM_PREC_FP64, nat.dptr(dr),
                                 nat.dptr(dv), nat.dptr(dt), sweeps, tol, every, ctypes.byref(done),
                                 ctypes.byref(delta))
    return rc, dv.cpu().numpy(), done.value, delta.value


def _inputs(shape, seed=5):
    from oracle import jacobi as oj
    rng = numpy.random.default_rng(seed)
    n = shape[0] * shape[1] * shape[2]
    return rng.standard_normal(n), numpy.where(oj.boundary_mask(*shape), rng.standard_normal(n), 0.0)


@pytest.mark.parametrize("n", [3, 4, 17, 18, 19, 34, 130, 131, 257, 258, 259, 514, 515, 1026, 1027])
@pytest.mark.parametrize("axis", [0, 1, 2])
def test_fixed_sweeps_along_each_axis(n, axis):
    """1 .. 1025 interior points along one axis (1025: left to the sweeps); the gate of the FP64 sweeps, 1e-12."""
    from oracle import jacobi as oj
    shape = [9, 7, 8]
    shape[axis] = n
    rho, v0 = _inputs(shape)
    print("[case] closed form", shape, flush=True)
    rc, got, done, _ = _jacobi(shape, rho, v0, 131)
    want = oj.jacobi(rho, *shape, 0.3, 131, bvals=v0, v0=v0)
    assert rc == 0 and done == 131
    assert numpy.abs(got - want).max() <= 1e-12 * numpy.abs(want).max()


@pytest.mark.parametrize("shape", [(24, 17, 20), (40, 12, 31)])
def test_check_stops_at_the_first_one_below_tolerance(shape):
    """The bisected check is the first whose delta, from plain sweeps, is at most the tolerance."""
    from oracle import jacobi as oj
    rho, v0 = _inputs(shape, 8)
    print("[case] closed form check", shape, flush=True)
    v, deltas = v0, []
    for _ in range(30):
        v = oj.jacobi(rho, *shape, 0.3, 39, bvals=v0, v0=v)
        t = oj.sweep(v, rho, *shape, 0.3, v0)
        deltas.append(float(numpy.abs(t - v).sum()))
        v = t
    for c in (0, 3, 17, 29):
        tol = deltas[c] * 1.0001
        rc, got, done, delta = _jacobi(shape, rho, v0, 40 * 30, tol, 40)
        assert rc == 0 and done == 40 * (c + 1)
        assert delta == pytest.approx(deltas[c], rel=1e-9)
        want = oj.jacobi_closed_form(rho, *shape, 0.3, done, bvals=v0)
        assert numpy.abs(got - want).max() <= 1e-12 * numpy.abs(want).max()


def test_values_that_are_not_finite_stay_local():
    """A NaN charge spreads one point per sweep, as with plain sweeps."""
    shape = (120, 8, 8)
    rho, v0 = _inputs(shape)
    rho[60 + 120 * (4 + 8 * 4)] = numpy.nan
    print("[case] closed form, NaN", flush=True)
    rc, got, done, _ = _jacobi(shape, rho, v0, 45)
    row = got.reshape(8, 8, 120)[4, 4]
    assert rc == 0 and done == 45
    assert numpy.isnan(row[60 - 44:60 + 45:2]).all()
    assert numpy.isfinite(row[:60 - 46]).all() and numpy.isfinite(row[60 + 46:]).all()


def test_charges_near_the_end_of_the_range():
    """Charges whose transform overflows while the relaxed field does not (here by a factor of 50)."""
    from oracle import jacobi as oj
    shape = (64, 64, 64)
    rho = numpy.full(64 ** 3, -1.8e305)
    v0 = numpy.zeros_like(rho)
    want = oj.jacobi(rho, *shape, 0.3, 131, bvals=v0, v0=v0)
    assert numpy.isfinite(want).all()
    print("[case] closed form, huge charges", flush=True)
    rc, got, done, _ = _jacobi(shape, rho, v0, 131)
    assert rc == 0 and done == 131
    assert numpy.abs(got - want).max() <= 1e-12 * numpy.abs(want).max()


@pytest.mark.parametrize("adsorb,diff,tol,maxiters", [(0.1, 0.01, 1e-9, None), (0.05, 0.02, 1e-9, None),
                                                      (0.05, 0.02, 1e-6, 400.5), (0.02, 0.02, 1e-6, 40),
                                                      (0.4, 0.05, 1e-9, None), (0.05, 0.02, -1.0, 24)])
@pytest.mark.parametrize("shape", [(24, 16, 40), (19, 33, 18)])
def test_vne_pairs_and_field(shape, adsorb, diff, tol, maxiters):
    """The pair count, convergence and field of the plain loop, in and out of the closed form's parameter range
    (ADS = DIF grows; DIF = 0.05 with ADS = 0.4 leaves a negative self weight); 1e-12, the sweeps' gate."""
    import torch
    import qmtools
    from conftest import BASIS
    from oracle import vne as ov
    from qmtools import _native as nat, synth
    from qmtools.qmtools import device_molecule
    mol = synth.synthetic_molecule(6, 3, qmtools.BasisSet(BASIS))
    h = 0.5
    o = mol.coords.mean(0) - 0.5 * h * numpy.array(shape)
    n = shape[0] * shape[1] * shape[2]
    cap = 10 * n ** (1.0 / 3) if maxiters is None else maxiters
    print("[case] vne closed form", shape, adsorb, diff, tol, cap, flush=True)
    v = torch.empty(n, dtype=torch.float64, device="cuda")
    t = torch.empty_like(v)
    pairs, delta, conv = ctypes.c_int64(0), ctypes.c_double(0), ctypes.c_int(0)
    nat.call("qm_vne_diffusion", device_molecule(mol).handle, nat.stream(),
             ctypes.byref(nat.geom((*shape, h, tuple(o)))), nat.QM_F64, adsorb, diff, tol, float(cap), nat.dptr(v),
             nat.dptr(t), ctypes.byref(pairs), ctypes.byref(delta), ctypes.byref(conv))
    want, wp, wd, wc = ov.vne_diffusion(mol.types, mol.coords, *shape, h, o, adsorb, diff, tol, cap)
    assert pairs.value == wp and bool(conv.value) == wc
    assert delta.value == pytest.approx(wd, rel=1e-6)
    got = v.cpu().numpy().reshape(want.shape)
    assert numpy.abs(got - want).max() <= 1e-12 * numpy.abs(want).max()
