"""Closed forms of the relaxations against the stream order that the C interface promises."""
import ctypes

import numpy
import pytest

pytestmark = pytest.mark.gpu


def _charge(shape, seed):
    import torch
    g = torch.Generator(device="cpu").manual_seed(seed)
    return torch.randn(shape[0] * shape[1] * shape[2], dtype=torch.float64, generator=g).cuda()


def _jacobi(stream, shape, rho, v, tmp, sweeps, tol=-1.0, every=0):
    from qmtools import _native as nat
    done, delta = ctypes.c_int64(0), ctypes.c_double(0)
    rc = nat.library().qm_jacobi(nat.context(), ctypes.c_void_p(stream.cuda_stream),
                                 ctypes.byref(nat.geom((*shape, 0.3, (0.0, 0.0, 0.0)))), nat.QM_PREC_FP64,
                                 nat.dptr(rho), nat.dptr(v), nat.dptr(tmp), sweeps, tol, every, ctypes.byref(done),
                                 ctypes.byref(delta))
    assert rc in (nat.QM_OK, nat.QM_ENOCONV)   # a cap reached first is an outcome too
    return done.value


def test_jacobi_with_a_tolerance_returns_finished():
    """With a tolerance the outcome goes to host scalars, so nothing is left on the stream at the return."""
    import torch
    shape = (256, 256, 256)
    rho = _charge(shape, 1)
    v, tmp = torch.zeros_like(rho), torch.empty_like(rho)
    s = torch.cuda.Stream()
    print("[case] tolerance, stream idle at return", flush=True)
    with torch.cuda.stream(s):
        for _ in range(2):
            v.zero_()
            torch.cuda.synchronize()
            _jacobi(s, shape, rho, v, tmp, 4000, 1e3, 40)
            assert s.query()


def test_vne_returns_finished():
    """qm_vne_diffusion synchronises its stream."""
    import torch
    import qmtools
    from conftest import BASIS
    from qmtools import _native as nat, synth
    from qmtools.qmtools import device_molecule
    mol = synth.synthetic_molecule(6, 3, qmtools.BasisSet(BASIS))
    shape, h = (256, 256, 256), 0.1
    o = mol.coords.mean(0) - 0.5 * h * numpy.array(shape)
    v = torch.empty(shape[0] * shape[1] * shape[2], dtype=torch.float64, device="cuda")
    t = torch.empty_like(v)
    handle = device_molecule(mol).handle
    s = torch.cuda.Stream()
    pairs, delta, conv = ctypes.c_int64(0), ctypes.c_double(0), ctypes.c_int(0)
    print("[case] V_ne, stream idle at return", flush=True)
    for _ in range(2):
        torch.cuda.synchronize()
        nat.call("qm_vne_diffusion", handle, ctypes.c_void_p(s.cuda_stream), ctypes.byref(nat.geom((*shape, h, tuple(o)))),
                 nat.QM_F64, 0.05, 0.02, 1e-6, 100.0, nat.dptr(v), nat.dptr(t), ctypes.byref(pairs),
                 ctypes.byref(delta), ctypes.byref(conv))
        assert s.query()


@pytest.mark.parametrize("other", ["fixed", "tolerance", "fp32", "vne"])
def test_calls_on_two_streams_of_one_context(other):
    """A fixed-count relaxation in flight on one stream and another call on a second one: the bits of either alone."""
    import torch
    import qmtools
    from conftest import BASIS
    from qmtools import _native as nat, synth
    from qmtools.qmtools import device_molecule
    mol = synth.synthetic_molecule(4, 3, qmtools.BasisSet(BASIS))
    handle = device_molecule(mol).handle
    big, small = (200, 190, 180), (40, 66, 34)
    rb, rs = _charge(big, 2), _charge(small, 3)

    def first(s):
        v = torch.zeros_like(rb)
        t = torch.empty_like(rb)
        torch.cuda.synchronize()
        return v, t, lambda: _jacobi(s, big, rb, v, t, 500)

    def second(s):
        v = torch.zeros_like(rs)
        t = torch.empty_like(rs)
        torch.cuda.synchronize()
        if other == "vne":
            g = nat.geom((*small, 0.5, tuple(mol.coords.mean(0) - 0.25 * numpy.array(small))))
            p, d, c = ctypes.c_int64(0), ctypes.c_double(0), ctypes.c_int(0)
            return v, t, lambda: nat.call("qm_vne_diffusion", handle, ctypes.c_void_p(s.cuda_stream), ctypes.byref(g),
                                          nat.QM_F64, 0.05, 0.02, 1e-7, 400.0, nat.dptr(v), nat.dptr(t),
                                          ctypes.byref(p), ctypes.byref(d), ctypes.byref(c))
        if other == "fp32":
            d, n = ctypes.c_double(0), ctypes.c_int64(0)
            return v, t, lambda: nat.call("qm_jacobi", ctypes.c_void_p(s.cuda_stream),
                                          ctypes.byref(nat.geom((*small, 0.3, (0.0, 0.0, 0.0)))), nat.QM_PREC_FP32,
                                          nat.dptr(rs), nat.dptr(v), None, 500, -1.0, 50, ctypes.byref(n),
                                          ctypes.byref(d))
        tol = (1e-3, 40) if other == "tolerance" else (-1.0, 0)
        return v, t, lambda: _jacobi(s, small, rs, v, t, 700, *tol)

    sa, sb = torch.cuda.Stream(), torch.cuda.Stream()
    want = []
    for make, s in ((first, sa), (second, sb)):
        v, _, run = make(s)
        run()
        torch.cuda.synchronize()
        want.append(v.cpu().numpy())
    print("[case] two streams, one context:", other, flush=True)
    for order in (0, 1, 0, 1):
        va, _ta, ra = first(sa)
        vb, _tb, rb2 = second(sb)
        for run in ((ra, rb2) if order == 0 else (rb2, ra)):
            run()
        torch.cuda.synchronize()
        assert numpy.array_equal(va.cpu().numpy(), want[0])
        assert numpy.array_equal(vb.cpu().numpy(), want[1])


def test_a_fixed_count_does_not_wait_for_the_stream():
    """Without a tolerance the call returns with its work queued: what ran on the stream before is still running."""
    import torch
    shape = (96, 80, 72)
    rho = _charge(shape, 5)
    v, tmp = torch.zeros_like(rho), torch.empty_like(rho)
    s = torch.cuda.Stream()
    a = torch.randn(8192, 8192, device="cuda")
    b = torch.empty_like(a)
    print("[case] fixed count, stream busy at return", flush=True)
    with torch.cuda.stream(s):
        torch.mm(a, a, out=b)
        _jacobi(s, shape, rho, v, tmp, 500)   # workspaces and tables exist from here on
        torch.cuda.synchronize()
        v.zero_()
        for _ in range(40):
            torch.mm(a, a, out=b)
        busy = torch.cuda.Event()
        busy.record(s)
        _jacobi(s, shape, rho, v, tmp, 500)
        waited = busy.query()
    torch.cuda.synchronize()
    assert not waited
    want = torch.zeros_like(rho)
    _jacobi(torch.cuda.current_stream(), shape, rho, want, tmp, 500)
    torch.cuda.synchronize()
    assert numpy.array_equal(v.cpu().numpy(), want.cpu().numpy())
