"""Block tiles of the density contractions (8 x 4 x 4 voxels, lists of active function groups) at their edges:
grids smaller than a tile, part-filled edge tiles, sub-points, tiles with no active group, the shell order."""
import ctypes

import numpy
import pytest
from conftest import BASIS

pytestmark = pytest.mark.gpu


def _system(mol):
    from oracle.basisfile import read_basis
    from oracle.system import make_system
    return make_system(mol.types, mol.coords, mol.dm, read_basis(BASIS))


def _raw(mol, geom, subgrid, prec):
    import torch
    from qmtools import _native as nat
    from qmtools.qmtools import device_molecule
    out = torch.full((geom[0] * geom[1] * geom[2],), float("nan"), dtype=torch.float64, device="cuda")
    nat.call("qm_density", device_molecule(mol).handle, nat.stream(), ctypes.byref(nat.geom(geom)), subgrid, prec,
             nat.QM_F64, nat.dptr(out), 0, None)
    return out.cpu().numpy()


@pytest.mark.parametrize("shape", [(1, 1, 1), (7, 3, 5), (8, 4, 4), (9, 4, 5), (33, 2, 17), (17, 21, 6)])
@pytest.mark.parametrize("natoms,subgrid", [(1, 1), (1, 3), (12, 1), (30, 2)])
def test_block_tiles_ragged(shape, natoms, subgrid):
    """The same gates as on full grids: 1e-10 (FP64), 1e-6 (split) of the largest value."""
    import qmtools
    from oracle import density as od
    from qmtools import _native as nat, synth
    mol = synth.synthetic_molecule(natoms, 6, qmtools.BasisSet(BASIS))
    h = 0.7
    o = mol.coords.mean(0) - 0.5 * h * numpy.array(shape) + 0.1
    print("[case] block tiles", shape, natoms, subgrid, flush=True)
    want = od.density_grid_raw(_system(mol), *shape, h, o, subgrid)
    for prec, tol in ((nat.QM_PREC_FP64, 1e-10), (nat.QM_PREC_F16X3, 1e-6)):
        got = _raw(mol, (*shape, h, tuple(o)), subgrid, prec)
        assert numpy.abs(got - want).max() <= tol * numpy.abs(want).max()


def test_block_tiles_without_active_groups():
    """A grid whose far tiles are beyond every cutoff: exactly zero there, the oracle's values elsewhere."""
    import qmtools
    from oracle import density as od
    from qmtools import _native as nat, synth
    mol = synth.synthetic_molecule(4, 9, qmtools.BasisSet(BASIS))
    shape, h = (80, 5, 4), 1.0
    o = mol.coords.mean(0) - 2.0
    print("[case] block tiles, inactive", flush=True)
    want = od.density_grid_raw(_system(mol), *shape, h, o, 1)
    for prec, tol in ((nat.QM_PREC_FP64, 1e-10), (nat.QM_PREC_F16X3, 1e-6)):
        got = _raw(mol, (*shape, h, tuple(o)), 1, prec)
        assert numpy.abs(got - want).max() <= tol * numpy.abs(want).max()
        assert (got.reshape(4, 5, 80)[:, :, 40:] == 0.0).all()


def test_basis_points_in_the_callers_order():
    """qm_basis_points writes rows in the caller's function order, whatever the internal shell order."""
    import torch
    import qmtools
    from oracle import density as od
    from qmtools import _native as nat, synth
    from qmtools.qmtools import device_molecule
    mol = synth.synthetic_molecule(9, 4, qmtools.BasisSet(BASIS))
    pts = numpy.random.default_rng(3).normal(size=(70, 3)) * 3.0
    want = od.basis_on_points(_system(mol), pts).T
    d = torch.tensor(pts.ravel(), device="cuda")
    phi = torch.empty(mol.nbf * 70, dtype=torch.float64, device="cuda")
    nat.call("qm_basis_points", device_molecule(mol).handle, nat.stream(), nat.dptr(d), 70, nat.dptr(phi))
    got = phi.cpu().numpy().reshape(mol.nbf, 70)
    assert numpy.abs(got - want).max() <= 1e-13 * numpy.abs(want).max()


@pytest.mark.parametrize("shape", [(88, 372, 4), (128, 32, 32), (121, 65, 37), (256, 128, 128), (256, 129, 128)])
def test_block_tiles_sorted_launches(shape):
    """1023 tiles (as numbered), 1024, 2720 and 32768 (by list length), 33792 (as numbered); the gates of the full
    grids on z slabs of 4 planes."""
    import qmtools
    from oracle import density as od
    from qmtools import _native as nat, synth
    mol = synth.synthetic_molecule(3, 12, qmtools.BasisSet(BASIS))
    h = 0.2
    o = mol.coords.mean(0) - 0.5 * h * numpy.array(shape) + 0.05
    nx, ny, nz = shape
    system = _system(mol)
    slabs = {k: od.density_grid_raw(system, nx, ny, 4, h, o + numpy.array([0, 0, k * h]), 1).reshape(4, ny, nx)
             for k in {0, (nz // 2) // 4 * 4, nz - 4}}
    top = max(numpy.abs(w).max() for w in slabs.values())
    print("[case] sorted tiles", shape, flush=True)
    for prec, tol in ((nat.QM_PREC_FP64, 1e-10), (nat.QM_PREC_F16X3, 1e-6)):
        got = _raw(mol, (*shape, h, tuple(o)), 1, prec).reshape(nz, ny, nx)
        assert numpy.isfinite(got).all()
        for k, want in slabs.items():
            assert numpy.abs(got[k:k + 4] - want).max() <= tol * top


@pytest.mark.parametrize("nbf,limit", [(65536, False), (65537, True)])
@pytest.mark.parametrize("prec", ["QM_PREC_F16X3", "QM_PREC_BF16X3", "QM_PREC_FP64"])
def test_basis_beyond_the_lists_of_the_split_path(nbf, limit, prec):
    """A tile's list holds 2048 groups of 32 functions: the split path refuses a larger basis before it looks for a
    density matrix, single and batched (FP64 takes larger ones; here the matrix is missing)."""
    import torch
    from qmtools import _native as nat
    zero, one = numpy.zeros(nbf, dtype=numpy.int32), numpy.ones(nbf, dtype=numpy.int32)
    z, xyz, alpha = numpy.array([6], dtype=numpy.int32), numpy.zeros(3), numpy.ones(1)
    mol = ctypes.c_void_p()
    nat.call("qm_mol_create", 1, nat.i32p(z), nat.f64p(xyz), nbf, nat.i32p(zero), nat.i32p(zero), nat.i32p(one),
             nat.i32p(zero), 1, nat.f64p(alpha), nat.f64p(alpha), ctypes.byref(mol))
    lib, ctx = nat.library(), nat.context()
    print("[case] list limit", nbf, prec, flush=True)
    try:
        out = torch.zeros(512, dtype=torch.float64, device="cuda")
        g = nat.geom((8, 8, 8, 0.3, (0.0, 0.0, 0.0)))
        want = nat.QM_ELIMIT if limit and prec != "QM_PREC_FP64" else nat.QM_EINVAL
        p = getattr(nat, prec)
        assert lib.qm_density(ctx, mol, nat.stream(), ctypes.byref(g), 1, p, nat.QM_F64, nat.dptr(out), 0, None) == want
        outs = (ctypes.c_void_p * 1)(out.data_ptr())
        assert lib.qm_density_batch(ctx, nat.stream(), 1, (ctypes.c_void_p * 1)(mol.value), (nat.Geom * 1)(g), outs, p,
                                    nat.QM_F64, 0) == want
    finally:
        lib.qm_mol_destroy(ctx, mol)


@pytest.mark.parametrize("shape,subgrid", [((9, 6, 5), 3), ((8, 4, 4), 5), ((3, 2, 1), 16)])
@pytest.mark.parametrize("prec", ["QM_PREC_FP64", "QM_PREC_F16X3"])
def test_sub_points_beyond_the_workspace_budget(shape, subgrid, prec):
    """A budget of 1 MiB holds 4 (FP64) or 9 (split) row tiles of 199 functions, fewer than one tile's sub-points:
    the workspaces stay within it and the bits are those of the whole tile at once."""
    import torch
    import qmtools
    from qmtools import _native as nat, synth
    from qmtools.qmtools import device_molecule
    mol = synth.synthetic_molecule(20, 6, qmtools.BasisSet(BASIS))
    h = 0.7
    o = mol.coords.mean(0) - 0.5 * h * numpy.array(shape) + 0.1
    want = _raw(mol, (*shape, h, tuple(o)), subgrid, getattr(nat, prec))
    handle = device_molecule(mol).handle
    print("[case] sub-point chunks", shape, subgrid, prec, mol.nbf, flush=True)
    ctx = nat.new_context()
    try:
        nat.call_ctx(ctx, "qm_tune_set", nat.QM_TUNE_PHI_MIB, 1)
        got = torch.full((want.size,), float("nan"), dtype=torch.float64, device="cuda")
        nat.call_ctx(ctx, "qm_density", handle, nat.stream(), ctypes.byref(nat.geom((*shape, h, tuple(o)))), subgrid,
                     getattr(nat, prec), nat.QM_F64, nat.dptr(got), 0, None)
        assert numpy.array_equal(got.cpu().numpy(), want)
        held = ctypes.c_int64(0)
        nat.library().qm_ctx_memory(ctx, ctypes.byref(held))
        assert held.value <= (1 << 20) * 5 // 4   # partial sums: an eighth of the basis values at most
    finally:
        nat.destroy_context(ctx)


def _best_ms(run, reps=6):
    import torch
    best = 1e9
    for _ in range(reps):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        run()
        b.record()
        b.synchronize()
        best = min(best, a.elapsed_time(b))
    return best


def _density_call(mol, geom, subgrid, prec):
    import torch
    from qmtools import _native as nat
    from qmtools.qmtools import device_molecule
    handle, g = device_molecule(mol).handle, nat.geom(geom)
    out = torch.empty(geom[0] * geom[1] * geom[2], dtype=torch.float64, device="cuda")
    return lambda: nat.call("qm_density", handle, nat.stream(), ctypes.byref(g), subgrid, prec, nat.QM_F64, nat.dptr(out),
                            0, None)


def test_sub_points_cost_what_their_grid_costs():
    """16^3 voxels of 4^3 sub-points are the points of 64^3 voxels: no more than 1.8 times their time."""
    import qmtools
    from qmtools import _native as nat, synth
    mol = synth.synthetic_molecule(12, 3, qmtools.BasisSet(BASIS))
    o = tuple(mol.coords.mean(0) - 9.0)
    print("[case] sub-points, time", flush=True)
    sub = _best_ms(_density_call(mol, (16, 16, 16, 18.0 / 16, o), 4, nat.QM_PREC_FP64))
    fine = _best_ms(_density_call(mol, (64, 64, 64, 18.0 / 64, o), 1, nat.QM_PREC_FP64))
    assert sub <= 1.8 * fine


THIN = [(1, 1, 300), (1, 300, 1), (300, 1, 1), (40, 37, 1), (1, 40, 37), (37, 1, 40), (2, 70, 9), (70, 3, 9), (9, 70, 2),
        (5, 1, 1), (3, 3, 3)]


@pytest.mark.parametrize("shape", THIN)
@pytest.mark.parametrize("subgrid", [1, 2])
def test_tiles_of_thin_grids(shape, subgrid):
    """Tiles that follow a thin grid's shape; the gates of the full grids, single and (one sub-point) batched."""
    import torch
    import qmtools
    from oracle import density as od
    from qmtools import _native as nat, synth
    from qmtools.qmtools import device_molecule
    mol = synth.synthetic_molecule(7, 6, qmtools.BasisSet(BASIS))
    h = 0.4
    o = mol.coords.mean(0) - 0.5 * h * numpy.array(shape) + 0.1
    print("[case] thin tiles", shape, subgrid, flush=True)
    want = od.density_grid_raw(_system(mol), *shape, h, o, subgrid)
    top = numpy.abs(want).max()
    for prec, tol in ((nat.QM_PREC_FP64, 1e-10), (nat.QM_PREC_F16X3, 1e-6)):
        got = _raw(mol, (*shape, h, tuple(o)), subgrid, prec)
        assert numpy.abs(got - want).max() <= tol * top
        if subgrid > 1:
            continue
        out = torch.full((want.size,), float("nan"), dtype=torch.float64, device="cuda")
        g = (nat.Geom * 1)(nat.geom((*shape, h, tuple(o))))
        nat.call("qm_density_batch", nat.stream(), 1, (ctypes.c_void_p * 1)(device_molecule(mol).handle), g,
                 (ctypes.c_void_p * 1)(out.data_ptr()), prec, nat.QM_F64, 0)
        assert numpy.abs(out.cpu().numpy() - want).max() <= tol * top


@pytest.mark.parametrize("shape", [(1, 1, 3072), (3072, 1, 1), (64, 48, 1)])
def test_thin_grids_cost_what_a_box_costs(shape):
    """3072 voxels of 2^3 sub-points on a line or plane across the molecule: at most three times a box of as many."""
    import qmtools
    from qmtools import _native as nat, synth
    mol = synth.synthetic_molecule(12, 3, qmtools.BasisSet(BASIS))
    print("[case] thin tiles, time", shape, flush=True)

    def best(sh):
        h = 18.0 / max(sh)
        o = tuple(mol.coords.mean(0) - 0.5 * h * numpy.array(sh))
        return _best_ms(_density_call(mol, (*sh, h, o), 2, nat.QM_PREC_FP64))
    assert best(shape) <= 3.0 * best((16, 16, 12))


@pytest.mark.parametrize("shape", [(128, 32, 32), (121, 65, 37)])
@pytest.mark.parametrize("natoms,prec", [(13, "QM_PREC_FP64"), (50, "QM_PREC_FP64"), (50, "QM_PREC_F16X3")])
def test_sorted_launches_of_larger_bases(natoms, prec, shape):
    """1024 and 2720 tiles of 8 and more groups (FP64) or 16 and more (split), taken by list length: the bits of
    launches of fewer than 1024 tiles, which are taken as numbered."""
    import qmtools
    from qmtools import _native as nat, autotune, synth
    mol = synth.synthetic_molecule(natoms, 12, qmtools.BasisSet(BASIS))
    assert mol.nbf > (112 if prec == "QM_PREC_FP64" else 480)
    h = 0.25
    o = mol.coords.mean(0) - 0.5 * h * numpy.array(shape) + 0.05
    print("[case] sorted tiles, larger basis", natoms, mol.nbf, shape, prec, flush=True)
    got = _raw(mol, (*shape, h, tuple(o)), 1, getattr(nat, prec))
    old = autotune.get("phi_mib")
    autotune.set("phi_mib", 64)   # at least 131 072 bytes a tile: at most 512 tiles
    try:
        want = _raw(mol, (*shape, h, tuple(o)), 1, getattr(nat, prec))
    finally:
        autotune.set("phi_mib", old)
    assert numpy.isfinite(got).all() and numpy.array_equal(got, want)
