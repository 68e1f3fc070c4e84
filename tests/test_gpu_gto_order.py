"""The order in which the GTO potential takes a grid's nodes, and how it shares out the distributions."""
import ctypes

import numpy
import pytest
from conftest import BASIS

pytestmark = pytest.mark.gpu


def _molecule(natoms, seed=3):
    import qmtools
    from qmtools import synth
    return synth.synthetic_molecule(natoms, seed, qmtools.BasisSet(BASIS))


def _nodes(shape, h, o):
    k, j, i = numpy.meshgrid(*[numpy.arange(n) for n in shape[::-1]], indexing="ij")
    return numpy.array(o) + h * numpy.stack([i, j, k], axis=-1).reshape(-1, 3)


def _calls(mol, shape, h, o):
    """Launchers of the grid call and of the list call on its nodes, with their outputs."""
    import torch
    from qmtools import _native as nat
    from qmtools.qmtools import device_molecule
    handle = device_molecule(mol).handle
    n = shape[0] * shape[1] * shape[2]
    pts = torch.tensor(_nodes(shape, h, o).ravel(), device="cuda")
    a, b = (torch.full((n,), float("nan"), dtype=torch.float64, device="cuda") for _ in range(2))
    g = nat.geom((*shape, h, tuple(o)))

    def grid():
        nat.call("qm_hartree_gto_grid", handle, nat.stream(), ctypes.byref(g), nat.QM_F64, nat.dptr(a))

    def points():
        nat.call("qm_hartree_gto_points", handle, nat.stream(), nat.dptr(pts), n, nat.dptr(b))
    return grid, points, a, b


@pytest.mark.parametrize("shape", [(1, 1, 1), (700, 1, 1), (1, 513, 1), (1, 1, 300), (40, 40, 1), (9, 9, 9), (64, 8, 8),
                                   (63, 8, 8), (61, 8, 8), (40, 48, 47), (40, 48, 44)])
def test_grid_equals_its_nodes(shape):
    """Nodes in blocks (padding up to 1/20) and in order; the parity gate of the potential, 1e-10."""
    mol = _molecule(5)
    h = 0.4
    o = mol.coords.mean(0) - 0.5 * h * numpy.array(shape) + 0.05
    print("[case] gto order", shape, flush=True)
    grid, points, a, b = _calls(mol, shape, h, o)
    grid()
    points()
    a, b = a.cpu().numpy(), b.cpu().numpy()
    assert numpy.abs(a - b).max() <= 1e-10 * numpy.abs(b).max()


@pytest.mark.parametrize("shape", [(20000, 1, 1), (128, 128, 1)])
def test_thin_grids_cost_what_their_nodes_cost(shape):
    """A line or a plane takes no more time than the list of its nodes, within a factor of two."""
    import torch
    mol = _molecule(12)
    h = 12.0 / max(shape)
    o = mol.coords.mean(0) - 0.5 * h * numpy.array(shape)
    print("[case] gto thin grid", shape, flush=True)
    grid, points, _, _ = _calls(mol, shape, h, o)

    def time(run):
        best = 1e9
        for _ in range(6):
            e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            e0.record()
            run()
            e1.record()
            e1.synchronize()
            best = min(best, e0.elapsed_time(e1))
        return best
    assert time(grid) <= 2.0 * time(points)


@pytest.mark.parametrize("natoms", [1, 2, 5, 7, 9])
@pytest.mark.parametrize("npts", [1, 700, 5000])
def test_shares_of_the_distributions(natoms, npts):
    """Few distributions and few points: chunks of equal cost over all lists (1 to 64 of them); the gate, 1e-10."""
    import torch
    from oracle import gto as og
    from oracle.basisfile import read_basis
    from oracle.system import make_system
    from qmtools import _native as nat
    from qmtools.qmtools import device_molecule
    mol = _molecule(natoms)
    pts = mol.coords.mean(0) + numpy.random.default_rng(natoms).uniform(-6, 6, size=(npts, 3))
    some = numpy.unique(numpy.r_[0:min(npts, 40), max(npts - 8, 0):npts])
    want = og.potential(make_system(mol.types, mol.coords, mol.dm, read_basis(BASIS)), pts[some])
    d = torch.tensor(pts.ravel(), device="cuda")
    out = torch.full((npts,), float("nan"), dtype=torch.float64, device="cuda")
    print("[case] gto shares", natoms, npts, flush=True)
    nat.call("qm_hartree_gto_points", device_molecule(mol).handle, nat.stream(), nat.dptr(d), npts, nat.dptr(out))
    got = out.cpu().numpy()
    assert numpy.isfinite(got).all()
    assert numpy.abs(got[some] - want).max() <= 1e-10 * numpy.abs(want).max()
