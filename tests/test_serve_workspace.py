"""The serving layer's estimate of a lane's workspaces against what the native density holds."""
import ctypes

import pytest
import qmtools
from conftest import BASIS
from qmtools import synth
from qmtools.serve import workspace_estimate


def _requests(count=2, n=48):
    basis = qmtools.BasisSet(BASIS)
    out = []
    for i in range(count):
        mol = synth.synthetic_molecule(13, i, basis)   # 128 functions
        grid = synth.centred_grid(mol, n, 0.3, 3.0)
        out.append(type("R", (), {"npts": int(grid.npts), "mol": mol, "grid": grid})())
    return out


@pytest.mark.parametrize("precision,per_point", [("fp64", 128 * 8 + 8 * 8 + 4), ("mixed", 128 * 4 + 2 * 8 + 4)])
def test_partial_densities_are_counted(precision, per_point):
    """Basis values, partial sums (8 groups of 16: one each; 4 groups of 32: two in all) and scales of a point."""
    reqs = _requests()
    npts = sum(r.npts for r in reqs)
    got = workspace_estimate(reqs, precision, "jacobi") - (0 if precision == "fp64" else 12 * npts)
    assert npts * per_point <= got <= npts * (per_point + 1)


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_density_batch_stays_within_the_estimate(precision):
    """A fresh lane holds at most the estimate after a density batch, and 64 KiB of small fixed tables."""
    from qmtools import _native as nat, batch
    reqs = _requests()
    lane = batch.Lane()
    print("[case] lane memory", precision, flush=True)
    try:
        batch.density_batch([r.mol for r in reqs], [r.grid for r in reqs], precision, lane=lane)
        lane.stream.synchronize()
        held = ctypes.c_int64(0)
        nat.check(nat.library().qm_ctx_memory(lane.ctx, ctypes.byref(held)), lane.ctx)
        assert held.value <= workspace_estimate(reqs, precision, "jacobi") + (1 << 16)
    finally:
        lane.close()
