"""Where the relaxations' closed forms hand a call back to the sweeps: the sweeps' own result, counts and bits."""
import ctypes

import numpy
import pytest

pytestmark = pytest.mark.gpu


def _state(shape, seed):
    import torch
    from oracle import jacobi as oj
    rng = numpy.random.default_rng(seed)
    n = shape[0] * shape[1] * shape[2]
    rho = rng.standard_normal(n)
    v = numpy.where(oj.boundary_mask(*shape), rng.standard_normal(n), 0.0)
    return torch.tensor(rho, device="cuda"), torch.tensor(v, device="cuda")


def _jacobi(shape, rho, v, sweeps, tol=-1.0, every=0, ctx=None):
    import torch
    from qmtools import _native as nat
    tmp = torch.empty_like(v)
    done, delta = ctypes.c_int64(0), ctypes.c_double(0)
    rc = nat.library().qm_jacobi(ctx or nat.context(), nat.stream(), ctypes.byref(nat.geom((*shape, 0.3, (0, 0, 0)))),
                                 nat.QM_PREC_FP64, nat.dptr(rho), nat.dptr(v), nat.dptr(tmp), sweeps, tol, every,
                                 ctypes.byref(done), ctypes.byref(delta))
    return rc, done.value, delta.value


def _loop(shape, rho, v, sweeps, tol, every):
    """The loop by calls of `every` sweeps, too few for the closed form."""
    assert every < 32
    for done in range(every, sweeps + 1, every):
        rc, _, delta = _jacobi(shape, rho, v, every, tol, every)
        if delta <= tol:
            break
    return rc, done, delta


@pytest.mark.parametrize("shape", [(12, 10, 9), (33, 6, 20)])
@pytest.mark.parametrize("tol", [1e-24, 0.0, 1e-11])
def test_tolerance_below_the_rounding_of_the_sweeps(shape, tol):
    """The public default, 1e-24, and 0 are decided by rounding on a small grid: the loop's field, sweep count and delta
    bit for bit.  1e-11 is above the floor of 1e-12 sum |V| on neither grid (sum |V| > 100)."""
    from qmtools import _native as nat
    rho, v0 = _state(shape, 4)
    want, got = v0.clone(), v0.clone()
    rw, nw, dw = _loop(shape, rho, want, 3000, tol, 30)
    assert float(want.abs().sum()) > 100
    print("[case] closed form, undecidable tolerance", shape, tol, nw, flush=True)
    rg, ng, dg = _jacobi(shape, rho, got, 3000, tol, 30)
    assert rg == rw and rg in (nat.QM_OK, nat.QM_ENOCONV)
    assert ng == nw and dg == dw
    assert numpy.array_equal(got.cpu().numpy(), want.cpu().numpy())


def test_vne_below_the_rounding_of_the_loop():
    """Pairs without a tolerance until their change is far below rounding (0.65^600): the loop's count and field."""
    import torch
    import qmtools
    from conftest import BASIS
    from oracle import vne as ov
    from qmtools import _native as nat, synth
    from qmtools.qmtools import device_molecule
    mol = synth.synthetic_molecule(6, 3, qmtools.BasisSet(BASIS))
    shape, h = (24, 16, 40), 0.5
    o = mol.coords.mean(0) - 0.5 * h * numpy.array(shape)
    v = torch.empty(shape[0] * shape[1] * shape[2], dtype=torch.float64, device="cuda")
    t = torch.empty_like(v)
    p, d, c = ctypes.c_int64(0), ctypes.c_double(0), ctypes.c_int(0)
    print("[case] V_ne closed form, undecidable", flush=True)
    nat.call("qm_vne_diffusion", device_molecule(mol).handle, nat.stream(),
             ctypes.byref(nat.geom((*shape, h, tuple(o)))), nat.QM_F64, 0.35, 0.02, -1.0, 300.0, nat.dptr(v),
             nat.dptr(t), ctypes.byref(p), ctypes.byref(d), ctypes.byref(c))
    want, wp, wd, wc = ov.vne_diffusion(mol.types, mol.coords, *shape, h, o, 0.35, 0.02, -1.0, 300.0)
    assert p.value == wp and bool(c.value) == wc
    assert 0.0 <= d.value <= 1e-15 * numpy.abs(want).max() and wd <= 1e-15 * numpy.abs(want).max()
    assert numpy.abs(v.cpu().numpy().reshape(want.shape) - want).max() <= 1e-12 * numpy.abs(want).max()


def test_under_stream_capture():
    """A captured call of 100 sweeps records the sweeps: every replay relaxes the buffer by 100 more.  (A context of its
    own: one that holds graphs of earlier calls asks for their events, which a capture does not allow.)"""
    import torch
    from qmtools import _native as nat
    shape = (40, 24, 19)
    rho, v0 = _state(shape, 6)
    want, v = v0.clone(), v0.clone()
    tmp = torch.empty_like(v)
    done, delta = ctypes.c_int64(0), ctypes.c_double(0)
    g = nat.geom((*shape, 0.3, (0, 0, 0)))
    graph = torch.cuda.CUDAGraph()
    ctx = nat.new_context()
    torch.cuda.synchronize()
    print("[case] closed form, capture", flush=True)
    try:
        with torch.cuda.graph(graph):
            nat.call_ctx(ctx, "qm_jacobi", nat.stream(), ctypes.byref(g), nat.QM_PREC_FP64, nat.dptr(rho), nat.dptr(v),
                         nat.dptr(tmp), 100, -1.0, 0, ctypes.byref(done), ctypes.byref(delta))
        for _ in range(3):
            for _ in range(5):
                _jacobi(shape, rho, want, 20)
            graph.replay()
            torch.cuda.synchronize()
            assert numpy.array_equal(v.cpu().numpy(), want.cpu().numpy())
    finally:
        nat.destroy_context(ctx)


@pytest.mark.parametrize("tol", [-1.0, 1e-6])
def test_no_room_for_the_tables(tol):
    """The sweeps need no workspace of the grid's size: where the sine tables cannot be had they run instead."""
    from qmtools import _native as nat
    shape = (530, 20, 24)
    rho, v0 = _state(shape, 7)
    want, got = v0.clone(), v0.clone()
    for _ in range(9):
        _jacobi(shape, rho, want, 20)
    print("[case] closed form, no room", tol, flush=True)
    ctx = nat.new_context()
    try:
        nat.call_ctx(ctx, "qm_tune_set", nat.QM_TUNE_WS_MIB, 1)
        rc, done, _ = _jacobi(shape, rho, got, 180, tol, 60, ctx)
        assert rc == (nat.QM_OK if tol < 0 else nat.QM_ENOCONV) and done == 180
        assert numpy.array_equal(got.cpu().numpy(), want.cpu().numpy())
    finally:
        nat.destroy_context(ctx)


def test_no_room_for_the_tables_of_vne():
    import torch
    import qmtools
    from conftest import BASIS
    from oracle import vne as ov
    from qmtools import _native as nat, synth
    from qmtools.qmtools import device_molecule
    mol = synth.synthetic_molecule(6, 3, qmtools.BasisSet(BASIS))
    shape, h = (530, 12, 10), 0.5
    o = mol.coords.mean(0) - 0.5 * h * numpy.array(shape)
    v = torch.empty(shape[0] * shape[1] * shape[2], dtype=torch.float64, device="cuda")
    t = torch.empty_like(v)
    p, d, c = ctypes.c_int64(0), ctypes.c_double(0), ctypes.c_int(0)
    handle = device_molecule(mol).handle
    print("[case] V_ne closed form, no room", flush=True)
    ctx = nat.new_context()
    try:
        nat.call_ctx(ctx, "qm_tune_set", nat.QM_TUNE_WS_MIB, 1)
        nat.call_ctx(ctx, "qm_vne_diffusion", handle, nat.stream(), ctypes.byref(nat.geom((*shape, h, tuple(o)))),
                     nat.QM_F64, 0.05, 0.02, 1e-7, 200.0, nat.dptr(v), nat.dptr(t), ctypes.byref(p), ctypes.byref(d),
                     ctypes.byref(c))
    finally:
        nat.destroy_context(ctx)
    want, wp, wd, wc = ov.vne_diffusion(mol.types, mol.coords, *shape, h, o, 0.05, 0.02, 1e-7, 200.0)
    assert p.value == wp and bool(c.value) == wc
    assert numpy.abs(v.cpu().numpy().reshape(want.shape) - want).max() <= 1e-12 * numpy.abs(want).max()


@pytest.mark.parametrize("tol,decided", [(1e2, True), (0.0, False)])
def test_profile_counts_the_sweeps_that_were_done(tol, decided):
    """A closed form that stops at a check counts as the sweeps up to it, one that is left to the sweeps as nothing."""
    from qmtools import _native as nat
    shape = (12, 10, 9)
    rho, v = _state(shape, 4)
    ctx = nat.new_context()
    print("[case] closed form, profile", tol, flush=True)
    try:
        nat.call_ctx(ctx, "qm_profile", 1)
        rc, done, _ = _jacobi(shape, rho, v, 3000, tol, 30, ctx)
        assert rc == nat.QM_OK and (done < 3000 or not decided)
        ms, n = ctypes.c_double(0), ctypes.c_int64(0)
        nat.call_ctx(ctx, "qm_profile_read", nat.QM_K_JACOBI, ctypes.byref(ms), ctypes.byref(n))
        assert n.value == done
    finally:
        nat.destroy_context(ctx)


@pytest.mark.parametrize("shape", [(3, 3, 3), (12, 10, 9), (70, 33, 20)])
@pytest.mark.parametrize("where", ["rho nan", "rho inf", "v inside", "v outside", "huge"])
@pytest.mark.parametrize("sweeps", [45, 80])
def test_residuals_left_to_the_sweeps(shape, where, sweeps):
    """Charges or values that are not finite, or too large for the transforms: the sweeps' bits, odd and even counts."""
    from qmtools import _native as nat
    rho, v0 = _state(shape, 8)
    nx, ny, nz = shape
    at = nx // 2 + nx * (ny // 2 + ny * (nz // 2))
    if where == "rho nan":
        rho[at] = float("nan")
    elif where == "rho inf":
        rho[at] = float("inf")
        rho[1 + nx * (1 + ny)] = float("-inf")
    elif where == "v inside":
        v0[at] = float("nan")
    elif where == "v outside":
        v0[nx // 2 + nx * (ny // 2)] = float("inf")
    else:
        rho[at] = 1e300
    want, got = v0.clone(), v0.clone()
    for q in range(0, sweeps, 20):
        _jacobi(shape, rho, want, min(20, sweeps - q))
    print("[case] left to the sweeps", shape, where, sweeps, flush=True)
    rc, done, _ = _jacobi(shape, rho, got, sweeps)
    assert rc == nat.QM_OK and done == sweeps
    numpy.testing.assert_array_equal(got.cpu().numpy(), want.cpu().numpy())
