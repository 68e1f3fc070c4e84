"""Timed cases of the grid hot path: density, Hartree potentials and the diffusion V_ne field.

Every case goes through the public entry points (`QMTools.Compute_*`, `qmtools.batch`) on seeded synthetic
molecules (C/N/O/H, cc-pVDZ, alpha-spin density matrix C C^T) and grids of the sizes that the benchmark, the
tests and the molecule cache use.  `exact` gives the same results in 64-bit torch, without the package's code.
"""
import math
import os
import sys

import numpy
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
for _p in (_ROOT, os.path.join(_ROOT, "qmtools-pycuda_amd")):
    if _p not in sys.path:
        sys.path.insert(0, _p)

import qmtools  # noqa: E402
from qmtools import batch, synth  # noqa: E402

ANG2BOR = 1.8897259886
SIGMA, CUTOFF = 0.2, 6.0


def listed():
    return [
        # the smallest call: one small molecule on a coarse grid, result on the host (smoke-test size);
        # launches, uploads and the copy back are what counts
        {"name": "density_fp64_5at_32", "kind": "density", "precision": "fp64", "atoms": 5, "nx": 32, "ny": 32,
         "nz": 32, "step": 0.3, "subgrid": 1, "host": True},
        # the molecule cache's ingest: two sub-points per axis on a box that follows the molecule's shape
        {"name": "density_fp64_24at_sub2", "kind": "density", "precision": "fp64", "atoms": 24, "nx": 104, "ny": 88,
         "nz": 72, "step": 0.19, "subgrid": 2, "host": False},
        # the headline workload, in both precisions
        {"name": "density_fp64_60at_256", "kind": "density", "precision": "fp64", "atoms": 60, "nx": 256, "ny": 256,
         "nz": 256, "step": 0.1, "subgrid": 1, "host": False},
        {"name": "density_mixed_60at_256", "kind": "density", "precision": "mixed", "atoms": 60, "nx": 256,
         "ny": 256, "nz": 256, "step": 0.1, "subgrid": 1, "host": False},
        # a batch of uneven molecules, density and free-space FFT Poisson in one call (whole pipeline)
        {"name": "batch_mixed_6mol_fft", "kind": "batch", "precision": "mixed", "count": 6, "atoms": 5,
         "atoms_max": 80, "n": 64, "n_max": 160, "step": 0.12},
        # Poisson relaxation of the headline grid: 2000 sweeps, open (multipole) boundaries
        {"name": "jacobi_fp64_256", "kind": "jacobi", "precision": "fp64", "atoms": 60, "nx": 256, "ny": 256,
         "nz": 256, "step": 0.1, "boundary": "multipole", "sweeps": 2000, "tolerance": 0.0, "host": False},
        # the same relaxation of a small molecule on the reduced-precision path (12 atoms, 96^3)
        {"name": "jacobi_mixed_12at_96", "kind": "jacobi", "precision": "mixed", "atoms": 12, "nx": 96, "ny": 96,
         "nz": 96, "step": 0.15, "boundary": "multipole", "sweeps": 2000, "tolerance": 0.0, "host": False},
        # relaxation to a tolerance with the reference's zero boundary on a ragged box, result on the host
        {"name": "jacobi_fp64_tol_ragged", "kind": "jacobi", "precision": "fp64", "atoms": 10, "nx": 72, "ny": 64,
         "nz": 56, "step": 0.25, "boundary": "zero", "sweeps": 100000, "tolerance": 1e-4, "host": True},
        # free-space FFT Poisson on a large box whose sides are no powers of two
        {"name": "fft_fp64_freespace", "kind": "fft", "precision": "fp64", "mode": "freespace", "atoms": 50,
         "nx": 240, "ny": 256, "nz": 200, "step": 0.12},
        # analytic potential at scattered points: the headline workload's third part
        {"name": "gto_points_60at", "kind": "gto", "where": "points", "atoms": 60, "points": 10000, "step": 0.1},
        # analytic potential at every node of a ragged box (the reference's Compute_hartree)
        {"name": "gto_grid_16at", "kind": "gto", "where": "grid", "atoms": 16, "nx": 48, "ny": 40, "nz": 56,
         "step": 0.4},
        # the molecule cache's second ingest step: diffusion V_ne to its default tolerance on a ragged box
        {"name": "vne_fp64_ragged", "kind": "vne", "precision": "fp64", "atoms": 12, "nx": 120, "ny": 120, "nz": 64,
         "adsorb": 0.05, "diff": 0.02, "step": 0.19},
    ]


def draw(rng):
    def side(lo, hi):
        return 8 * int(round(math.exp(rng.uniform(math.log(lo / 8), math.log(hi / 8)))))

    def box(lo, hi):
        return {"nx": side(lo, hi), "ny": side(lo, hi), "nz": side(lo, hi)}

    def atoms(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    step = round(rng.uniform(0.1, 0.3), 4)
    kind = rng.choice(["density", "density", "batch", "jacobi", "fft", "gto", "vne"])
    if kind == "density":
        sub = rng.choice([1, 1, 2])
        return {"kind": kind, "precision": rng.choice(["fp64", "mixed"]), "atoms": atoms(5, 60),
                **box(32, 224 if sub == 1 else 112), "step": step, "subgrid": sub, "host": rng.random() < 0.3}
    if kind == "batch":
        return {"kind": kind, "precision": rng.choice(["fp64", "mixed"]), "count": rng.randint(2, 6), "atoms": 5,
                "atoms_max": rng.randint(20, 80), "n": 64, "n_max": rng.choice([96, 128, 160]), "step": step}
    if kind == "jacobi":
        tol = rng.random() < 0.3
        return {"kind": kind, "precision": "fp64" if tol else rng.choice(["fp64", "mixed"]), "atoms": atoms(5, 60),
                **box(40, 72 if tol else 232), "step": step, "boundary": "zero" if tol else "multipole",
                "sweeps": 100000 if tol else 100 * rng.randint(3, 20), "tolerance": 1e-4 if tol else 0.0,
                "host": rng.random() < 0.3}
    if kind == "fft":
        return {"kind": kind, "precision": rng.choice(["fp64", "mixed"]), "mode": rng.choice(["freespace", "periodic"]),
                "atoms": atoms(5, 60), **box(48, 240), "step": step}
    if kind == "gto":
        if rng.random() < 0.5:
            return {"kind": kind, "where": "points", "atoms": atoms(5, 60),
                    "points": int(round(math.exp(rng.uniform(math.log(100), math.log(10000))))), "step": step}
        return {"kind": kind, "where": "grid", "atoms": atoms(3, 16), **box(24, 48), "step": step}
    return {"kind": kind, "precision": rng.choice(["fp64", "mixed"]), "atoms": atoms(5, 40), **box(48, 128),
            "adsorb": rng.choice([0.1, 0.05]), "diff": rng.choice([0.01, 0.02]), "step": step}


# ------------------------------------------------------------------ inputs
_BASIS = []


def _basis():
    if not _BASIS:
        _BASIS.append(qmtools.BasisSet(qmtools.basis.default_basis_path()))
    return _BASIS[0]


def _molecule(atoms, seed):
    for k in range(100):
        try:
            return synth.synthetic_molecule(atoms, (seed * 7919 + 31 * k + 5) % (1 << 31), _basis())
        except (ValueError, RuntimeError):   # a draw of elements that cannot carry the hydrogens
            continue
    raise RuntimeError("no molecule")


def _box_grid(mol, nx, ny, nz, step, dtype=numpy.float64):
    """Grid of the given shape centred on the molecule, step (bohr) grown until 2 Angstrom of padding fit."""
    lo, hi = mol.coords.min(0), mol.coords.max(0)
    n = numpy.array([nx, ny, nz], dtype=numpy.float64)
    h = max(step, float(((hi - lo + 4.0 * ANG2BOR) / n).max()))
    g = qmtools.Grid((1, nx, ny, nz), 1.0, dtype=dtype)
    g.step = numpy.float64(h)
    g.origin = qmtools.make_float3(*(0.5 * (lo + hi) - 0.5 * n * h))
    return g


def _axes(grid, shift):
    """Node (shift 0) or voxel-centre (shift 1/2) coordinates along x, y, z (bohr, FP64, on the GPU)."""
    nx, ny, nz, h, o = grid.geometry()
    return [o[d] + (torch.arange(n, dtype=torch.float64, device="cuda") + shift) * h
            for d, n in enumerate((nx, ny, nz))]


def _promolecule(mol, grid):
    """Electrons per voxel of superposed atomic densities (three Gaussians per atom), summing to sum Z:
    the charge that the Poisson solvers are given, flat x-fastest."""
    ax = _axes(grid, 0.5)
    widths, parts = [], []
    for z in mol.types:
        for a, f in ((0.35, 0.55), (1.4, 0.3), (1.1 * float(z), 0.15)):
            widths.append(a)
            parts.append(float(z) * f * (a / math.pi) ** 1.5)
    a = torch.tensor(widths, dtype=torch.float64, device="cuda")[:, None]
    w = torch.tensor(parts, dtype=torch.float64, device="cuda")[:, None]
    c = torch.tensor(numpy.repeat(mol.coords, 3, axis=0), device="cuda")
    ex, ey, ez = [torch.exp(-a * (x[None, :] - c[:, d, None]) ** 2) for d, x in enumerate(ax)]
    q = torch.empty((len(ax[2]), len(ax[1]), len(ax[0])), dtype=torch.float64, device="cuda")
    for k in range(q.shape[0]):
        q[k] = (ey * (w * ez[:, k:k + 1])).t().contiguous() @ ex
    q *= float(mol.qtot) / q.sum()
    return q.reshape(-1)


def _batch_items(case, seed):
    rng = numpy.random.default_rng(seed)
    mols, grids = [], []
    for i in range(case["count"]):
        # one molecule of every size class: the batch's work does not hang on the seed
        f = i / max(1, case["count"] - 1)
        na = int(round(case["atoms"] + f * (case["atoms_max"] - case["atoms"])))
        n = 8 * int(round((case["n_max"] + (1 - 2 * abs(f - 0.5)) * (case["n"] - case["n_max"])) / 8))
        mols.append(_molecule(na, seed * 64 + i))
        grids.append(synth.centred_grid(mols[-1], n, case["step"] + float(rng.uniform(0, 0.02)), 3.0))
    return mols, grids


def _points(mol, case, seed):
    lo, hi = mol.coords.min(0) - 3.0 * ANG2BOR, mol.coords.max(0) + 3.0 * ANG2BOR
    return lo + numpy.random.default_rng(seed).uniform(size=(case["points"], 3)) * (hi - lo)


def _inputs(case, seed):
    """Host molecule, grid and device charge of a case, from the seed alone."""
    if case["kind"] == "batch":
        return _batch_items(case, seed)
    mol = _molecule(case["atoms"], seed)
    if case["kind"] == "gto" and case["where"] == "points":
        return mol, _points(mol, case, seed), None
    dt = numpy.float32 if case.get("precision") == "mixed" and case["kind"] == "vne" else numpy.float64
    grid = _box_grid(mol, case["nx"], case["ny"], case["nz"], case["step"], dt)
    q = _promolecule(mol, grid) if case["kind"] in ("jacobi", "fft") else None
    return mol, grid, q


def prepare(case, seed):
    if case["kind"] == "batch":
        mols, grids = _batch_items(case, seed)
        for m in mols:
            m.upload()
        return {"case": case, "mols": mols, "grids": grids}
    mol, grid, q = _inputs(case, seed)
    mol.upload()
    state = {"case": case, "mol": mol, "grid": grid}
    if case["kind"] == "jacobi":
        state["qgrid"] = qmtools.Grid.emptyAs(grid)
        state["qgrid"].d_qube = q
    elif case["kind"] == "fft":
        state["q"] = q if case["precision"] == "fp64" else q.float()
    return state


def run(state):
    case = state["case"]
    kind = case["kind"]
    api = qmtools.QMTools
    if kind == "density":
        g = api.Compute_density(state["grid"], state["mol"], subgrid=case["subgrid"], copyBack=case["host"],
                                precision=case["precision"])
        return {"q": g.qube if case["host"] else g.d_qube, "raw_total": g.raw_total}
    if kind == "batch":
        qs, vs = batch.run(state["mols"], state["grids"], case["precision"], poisson="fft")
        return {"q": qs, "v": vs}
    if kind == "jacobi":
        tol = case["tolerance"]
        v = api.Compute_hartree_iter(state["qgrid"], state["mol"], tolerance=tol if tol > 0 else None,
                                     copyBack=case["host"], boundary=case["boundary"], max_sweeps=case["sweeps"],
                                     precision=case["precision"])
        return {"v": v.qube if case["host"] else v.d_qube, "sweeps": int(v.sweeps)}
    if kind == "fft":
        return batch.hartree_fft_batch([state["mol"]], [state["grid"]], [state["q"]], case["precision"],
                                       mode=case["mode"], sigma=SIGMA, cutoff=CUTOFF)[0]
    if kind == "gto":
        if case["where"] == "points":
            return api.Compute_hartree_points(state["mol"], state["grid"])
        api.Compute_hartree(state["grid"], state["mol"], copyBack=False)
        return state["grid"].d_qube
    v = api.Compute_VNe(state["grid"], state["mol"], adsorb=case["adsorb"], diff=case["diff"], copyBack=False,
                        precision=case["precision"])
    return {"v": v.d_qube, "pairs": int(v.pairs)}


# ------------------------------------------------------------------ the work of one pass
def _active(mol, pts):
    """Mean of n and n^2 over points, n = basis functions whose most diffuse primitive is above e^-50 there."""
    amin = numpy.array([mol.prim_alpha[p:p + k].min() for p, k in zip(mol.shell_poff, mol.shell_nprim)])
    nf = 2 * mol.shell_L + 1
    d2 = ((pts[:, None, :] - mol.coords[mol.shell_atom][None]) ** 2).sum(-1)
    n = ((d2 * amin[None, :] < 50.0) * nf[None, :]).sum(1).astype(numpy.float64)
    return n.mean(), (n * n).mean()


def _density_work(mol, grid, subgrid):
    nx, ny, nz, h, o = grid.geometry()
    pts = numpy.array(o) + numpy.random.default_rng(0).uniform(size=(400, 3)) * numpy.array([nx, ny, nz]) * h
    n1, n2 = _active(mol, pts)
    npts = float(nx * ny * nz) * subgrid ** 3
    # the triangle phi^T M phi plus the row-dot, over the functions that are not negligible at a point
    return npts * (n2 + 3.0 * n1), 8.0 * mol.nbf ** 2


def _fft_work(npts):
    # forward and inverse transform of the real padded box (8 x the points)
    m = 8.0 * npts
    return 2 * 2.5 * m * math.log2(m)


def _pairs(mol):
    """Primitive pairs (each exponent of an atom and L once) whose product is above 1e-17."""
    keys = {}
    for a, L, p, k in zip(mol.shell_atom, mol.shell_L, mol.shell_poff, mol.shell_nprim):
        for al in mol.prim_alpha[p:p + k]:
            keys[(int(a), int(L), float(al))] = 1
    at = numpy.array([k[0] for k in keys])
    al = numpy.array([k[2] for k in keys])
    d2 = ((mol.coords[at][:, None] - mol.coords[at][None]) ** 2).sum(-1)
    mu = al[:, None] * al[None] / (al[:, None] + al[None])
    return 0.5 * float((mu * d2 < 39.0).sum())


def work(case):
    kind = case["kind"]
    if kind == "batch":
        mols, grids = _batch_items(case, 1)
        b = f = 0.0
        size = 8 if case["precision"] == "fp64" else 4
        for m, g in zip(mols, grids):
            df, db = _density_work(m, g, 1)
            f += df + _fft_work(float(g.npts))
            b += db + 2.0 * size * float(g.npts)
        return {"bytes": b, "flops": f}
    mol = _molecule(case["atoms"], 1)
    if kind == "gto":
        n = case["points"] if case["where"] == "points" else case["nx"] * case["ny"] * case["nz"]
        # a Boys value, its recursion and the Hermite contraction: about 60 operations a pair and point
        return {"bytes": 32.0 * n if case["where"] == "points" else 8.0 * n, "flops": 60.0 * n * _pairs(mol)}
    npts = float(case["nx"] * case["ny"] * case["nz"])
    if kind == "density":
        f, b = _density_work(mol, _box_grid(mol, case["nx"], case["ny"], case["nz"], case["step"]), case["subgrid"])
        return {"bytes": b + npts * (8 if case["precision"] == "fp64" else 4), "flops": f}
    if kind == "fft":
        size = 8 if case["precision"] == "fp64" else 4
        return {"bytes": 2.0 * size * npts, "flops": _fft_work(npts)}
    if kind == "jacobi":   # charge in, potential out; a fixed sweep count has a closed form by sine transforms
        return {"bytes": 16.0 * npts, "flops": 6 * 2.5 * npts * math.log2(npts)}
    return {"bytes": (8.0 if case["precision"] == "fp64" else 4.0) * npts, "flops": 6 * 2.5 * npts * math.log2(npts)}


# ------------------------------------------------------------------ the same results in 64 bits
_C0, _C1, _C2A, _C20, _C22 = (0.28209479177387814, 0.4886025119029199, 1.0925484305920792, 0.31539156525252005,
                              0.5462742152960396)
_M_ORDER = {0: (0,), 1: (0, 1, -1), 2: (0, 1, -1, 2, -2)}
# Cartesian terms of the real solid harmonics: (coefficient, powers of x, y, z)
_CART = {(0, 0): [(_C0, (0, 0, 0))],
         (1, -1): [(_C1, (0, 1, 0))], (1, 0): [(_C1, (0, 0, 1))], (1, 1): [(_C1, (1, 0, 0))],
         (2, -2): [(_C2A, (1, 1, 0))], (2, -1): [(_C2A, (0, 1, 1))], (2, 1): [(_C2A, (1, 0, 1))],
         (2, 0): [(2 * _C20, (0, 0, 2)), (-_C20, (2, 0, 0)), (-_C20, (0, 2, 0))],
         (2, 2): [(_C22, (2, 0, 0)), (-_C22, (0, 2, 0))]}


def _total_dm(mol):
    return 2.0 * (numpy.tril(mol.dm) + numpy.tril(mol.dm, -1).T)


def _phi(mol, pts):
    """Basis values (nbf, n) at points (n, 3)."""
    out = torch.empty((mol.nbf, pts.shape[0]), dtype=torch.float64, device="cuda")
    f = 0
    for a, L, p, k in zip(mol.shell_atom, mol.shell_L, mol.shell_poff, mol.shell_nprim):
        d = pts - torch.tensor(mol.coords[a], device="cuda")
        r2 = (d * d).sum(1)
        rad = torch.zeros_like(r2)
        for al, co in zip(mol.prim_alpha[p:p + k], mol.prim_coeff[p:p + k]):
            rad += float(co) * torch.exp(-float(al) * r2)
        for m in _M_ORDER[int(L)]:
            ang = 0.0
            for c, e in _CART[(int(L), m)]:
                t = torch.full_like(r2, c)
                for ax in range(3):
                    for _ in range(e[ax]):
                        t = t * d[:, ax]
                ang = ang + t
            out[f] = ang * rad
            f += 1
    return out


def _exact_density(mol, grid, subgrid):
    nx, ny, nz, h, _ = grid.geometry()
    P = torch.tensor(_total_dm(mol), device="cuda")
    q = torch.zeros(nx * ny * nz, dtype=torch.float64, device="cuda")
    chunk = 1 << 18
    for sx in range(subgrid):
        for sy in range(subgrid):
            for sz in range(subgrid):
                x, y, z = [_axes(grid, (s + 0.5) / subgrid)[d] for d, s in enumerate((sx, sy, sz))]
                for t0 in range(0, q.numel(), chunk):
                    t = torch.arange(t0, min(t0 + chunk, q.numel()), device="cuda")
                    pts = torch.stack([x[t % nx], y[(t // nx) % ny], z[t // (nx * ny)]], 1)
                    f = _phi(mol, pts)
                    q[t0:t0 + chunk] += ((P @ f) * f).sum(0)
    q *= h ** 3 / subgrid ** 3
    total = q.sum()
    return q * (float(mol.qtot) / total), float(total)


def _exact_rhs(q, mol, grid):
    """Electrons per voxel and Gaussian nuclei as -rho_tot / eps0 (volt, Angstrom), array [i, j, k]."""
    nx, ny, nz, h, o = grid.geometry()
    s = h / ANG2BOR
    rhs = q.reshape(nz, ny, nx).permute(2, 1, 0).contiguous() / (-s ** 3)
    x, y, z = [o[d] / ANG2BOR + (torch.arange(n, dtype=torch.float64, device="cuda") + 0.5) * s
               for d, n in enumerate((nx, ny, nz))]
    norm = 1.0 / (SIGMA ** 3 * 2 * math.pi * math.sqrt(2 * math.pi))
    for zt, r in zip(mol.types, mol.coords * 0.529177211):
        r2 = ((x - r[0]) ** 2)[:, None, None] + ((y - r[1]) ** 2)[None, :, None] + ((z - r[2]) ** 2)[None, None, :]
        rhs += torch.where(r2 <= (CUTOFF * SIGMA) ** 2, float(zt) * norm * torch.exp(-r2 / (2 * SIGMA * SIGMA)), 0.0)
    return rhs / -0.0055263494, s


def _exact_fft(q, mol, grid, mode):
    rhs, s = _exact_rhs(q, mol, grid)
    shape = rhs.shape
    if mode == "periodic":
        k = [torch.fft.fftfreq(n, d=s, dtype=torch.float64, device="cuda") for n in shape]
        k2 = (k[0] ** 2)[:, None, None] + (k[1] ** 2)[None, :, None] + (k[2] ** 2)[None, None, :]
        f = torch.fft.fftn(rhs) * (-1.0 / (4 * math.pi ** 2 * k2))
        f[0, 0, 0] = 0.0
        return torch.fft.ifftn(f).real.contiguous().reshape(-1)
    dist = [torch.minimum(i, 2 * n - i).double() * s for n in shape for i in [torch.arange(2 * n, device="cuda")]]
    g = torch.sqrt((dist[0] ** 2)[:, None, None] + (dist[1] ** 2)[None, :, None] + (dist[2] ** 2)[None, None, :])
    g[0, 0, 0] = s / (2.0 * (3.0 * math.asinh(1.0 / math.sqrt(2.0)) - math.pi / 4.0))
    full = tuple(2 * n for n in shape)
    f = torch.fft.rfftn(1.0 / g) * torch.fft.rfftn(rhs, s=full)
    v = torch.fft.irfftn(f, s=full)[:shape[0], :shape[1], :shape[2]]
    return (v * (-s ** 3 / (4.0 * math.pi))).contiguous().reshape(-1)


def _seed(mol, grid):
    nx, ny, nz, h, o = grid.geometry()
    out = torch.zeros((nz, ny, nx), dtype=torch.float64)
    for zt, r in zip(mol.types, mol.coords):
        a = r - numpy.array(o)
        i0 = numpy.floor(a / h).astype(int)
        for c in range(8):
            i = i0 + numpy.array([c & 1, (c >> 1) & 1, c >> 2])
            if (i >= 0).all() and i[0] < nx and i[1] < ny and i[2] < nz:
                out[i[2], i[1], i[0]] = float(zt) * float(numpy.prod(numpy.abs(a - i * h) / h))
    return out.cuda()


def _multipole(rho, grid):
    """-phi/(4 pi) of the charges' monopole, dipole and quadrupole about the box centre, at every node."""
    nx, ny, nz, h, o = grid.geometry()
    n = (nx, ny, nz)
    x, y, z = [a - (o[d] + 0.5 * h * (n[d] - 1)) for d, a in enumerate(_axes(grid, 0.0))]
    X, Y, Z = x[None, None, :], y[None, :, None], z[:, None, None]
    q = rho.sum()
    p = [(rho * c).sum() for c in (X, Y, Z)]
    m2 = {(a, b): (rho * A * B).sum() for a, A in enumerate((X, Y, Z)) for b, B in enumerate((X, Y, Z)) if a <= b}
    tr = m2[(0, 0)] + m2[(1, 1)] + m2[(2, 2)]
    r2 = X * X + Y * Y + Z * Z
    r = torch.sqrt(r2)
    quad = sum((3.0 * v - (tr if a == b else 0.0)) * (1.0 if a == b else 2.0) * (X, Y, Z)[a] * (X, Y, Z)[b]
               for (a, b), v in m2.items())
    phi = q / r + (p[0] * X + p[1] * Y + p[2] * Z) / (r2 * r) + 0.5 * quad / (r2 * r2 * r)
    return phi / (-4.0 * math.pi)


def _sine(n):
    i = torch.arange(1, n + 1, dtype=torch.int64, device="cuda")
    k = (i[:, None] * i[None, :]) % (2 * (n + 1))
    return torch.sin(k.double() * (math.pi / (n + 1))) * math.sqrt(2.0 / (n + 1))


def _sine3(a, s):
    """Orthonormal sine transform (its own inverse) along the three axes of an array [z, y, x]."""
    a = a @ s[0]
    a = torch.matmul(s[1], a)
    return (s[2] @ a.reshape(a.shape[0], -1)).reshape(a.shape)


def _exact_jacobi(q, mol, grid, case):
    nx, ny, nz, h, _ = grid.geometry()
    rho = _seed(mol, grid) - q.reshape(nz, ny, nx)
    v = torch.zeros_like(rho)
    if case["boundary"] == "multipole":
        v = _multipole(rho, grid)
        v[1:-1, 1:-1, 1:-1] = 0.0
    c = (v[1:-1, 1:-1, :-2] + v[1:-1, 1:-1, 2:] + v[1:-1, :-2, 1:-1] + v[1:-1, 2:, 1:-1] + v[:-2, 1:-1, 1:-1]
         + v[2:, 1:-1, 1:-1] - rho[1:-1, 1:-1, 1:-1] / h) / 6.0
    s = [_sine(n - 2) for n in (nx, ny, nz)]
    hv = [torch.sin(torch.arange(1, n - 1, dtype=torch.float64, device="cuda") * (0.5 * math.pi / (n - 1))) ** 2
          for n in (nx, ny, nz)]
    one = (2.0 / 3.0) * (hv[0][None, None, :] + hv[1][None, :, None] + hv[2][:, None, None])   # 1 - eigenvalue
    mu = 1.0 - one
    ch = _sine3(c, s)

    def power(m):   # mu^m, accurate where mu is near 1
        return torch.where(one < 0.5, torch.exp(m * torch.log1p(-one.clamp(max=0.5))), mu ** m)

    m = case["sweeps"]
    if case["tolerance"] > 0:
        m = 200
        while float(_sine3(ch * power(m - 1), s).abs().sum()) > case["tolerance"]:
            m += 200
    geo = torch.where(one < 0.5, -torch.expm1(m * torch.log1p(-one.clamp(max=0.5))), 1.0 - mu ** m) / one
    v[1:-1, 1:-1, 1:-1] = _sine3(ch * geo, s)
    return v.reshape(-1), m


def _boys(top, T):
    """F_0 .. F_top: series and downward recursion below T = 8, erf and upward recursion above."""
    small = T < 8.0
    Ts = torch.where(small, T, 0.0)
    e = torch.exp(-Ts)
    term = torch.full_like(Ts, 1.0 / (2 * top + 1))
    ser = term.clone()
    for k in range(1, 60):
        term = term * Ts * (2.0 / (2 * top + 2 * k + 1))
        ser = ser + term
    low = [None] * (top + 1)
    low[top] = e * ser
    for n in range(top, 0, -1):
        low[n - 1] = (2 * Ts * low[n] + e) / (2 * n - 1)
    Tb = torch.where(small, 8.0, T)
    eb = torch.exp(-Tb)
    f = 0.5 * torch.sqrt(math.pi / Tb) * torch.erf(torch.sqrt(Tb))
    out = []
    for n in range(top + 1):
        out.append(torch.where(small, low[n], f))
        f = ((2 * n + 1) * f - eb) / (2 * Tb)
    return out


def _hermite_e(la, lb, a, b, ab):
    """Hermite expansion coefficients of one axis, E[i, j, t] over arrays of primitive pairs."""
    p = a + b
    E = {(0, 0, 0): numpy.exp(-a * b / p * ab * ab)}

    def get(i, j, t):
        return E.get((i, j, t), 0.0)
    for i in range(la + 1):
        for j in range(lb + 1):
            for t in range(i + j + 1):
                if i:
                    E[(i, j, t)] = get(i - 1, j, t - 1) / (2 * p) - b / p * ab * get(i - 1, j, t) + \
                        (t + 1) * get(i - 1, j, t + 1)
                elif j:
                    E[(i, j, t)] = get(i, j - 1, t - 1) / (2 * p) + a / p * ab * get(i, j - 1, t) + \
                        (t + 1) * get(i, j - 1, t + 1)
    return E


def _exact_gto(mol, pts):
    P = _total_dm(mol)
    prim = []   # shell, exponent, coefficient
    for s, (p, k) in enumerate(zip(mol.shell_poff, mol.shell_nprim)):
        prim += [(s, mol.prim_alpha[i], mol.prim_coeff[i]) for i in range(p, p + k)]
    sh = numpy.array([p[0] for p in prim])
    al = numpy.array([p[1] for p in prim])
    co = numpy.array([p[2] for p in prim])
    L = mol.shell_L[sh]
    X = mol.coords[mol.shell_atom[sh]]
    V = torch.zeros(pts.shape[0], dtype=torch.float64, device="cuda")
    for zt, r in zip(mol.types, mol.coords):
        d = torch.sqrt(((pts - torch.tensor(r, device="cuda")) ** 2).sum(1))
        V += torch.where(d > 1e-8, float(zt) / torch.where(d > 1e-8, d, 1.0), 0.0)
    for la in range(3):
        for lb in range(3):
            i, j = numpy.nonzero((L[:, None] == la) & (L[None] == lb) & (sh[:, None] >= sh[None]))
            if not len(i):
                continue
            a, b = al[i], al[j]
            ab = X[i] - X[j]
            keep = a * b / (a + b) * (ab ** 2).sum(1) < 45.0   # e^-45 of the overlap: below the last bit of the sum
            i, j, a, b, ab = i[keep], j[keep], a[keep], b[keep], ab[keep]
            p = a + b
            E = [_hermite_e(la, lb, a, b, ab[:, d]) for d in range(3)]
            pref = co[i] * co[j] * 2 * math.pi / p * numpy.where(sh[i] == sh[j], 1.0, 2.0)
            D = {}
            for ma, fa in enumerate(_M_ORDER[la]):
                for mb, fb in enumerate(_M_ORDER[lb]):
                    w = pref * P[mol.shell_bf[sh[i]] + ma, mol.shell_bf[sh[j]] + mb]
                    for ca, ea in _CART[(la, fa)]:
                        for cb, eb in _CART[(lb, fb)]:
                            for t in range(ea[0] + eb[0] + 1):
                                for u in range(ea[1] + eb[1] + 1):
                                    for v in range(ea[2] + eb[2] + 1):
                                        D[(t, u, v)] = D.get((t, u, v), 0.0) + ca * cb * w * \
                                            E[0][(ea[0], eb[0], t)] * E[1][(ea[1], eb[1], u)] * \
                                            E[2][(ea[2], eb[2], v)]
            D = {k: torch.tensor(v, device="cuda")[:, None] for k, v in D.items()}
            pt = torch.tensor(p, device="cuda")[:, None]
            C = torch.tensor((a[:, None] * X[i] + b[:, None] * X[j]) / p[:, None], device="cuda")
            top = la + lb
            rows = max(1, (1 << 25) // max(1, pts.shape[0]))
            for r0 in range(0, len(a), rows):
                sl = slice(r0, r0 + rows)
                d = [C[sl, ax, None] - pts[None, :, ax] for ax in range(3)]
                pp = pt[sl]
                F = _boys(top, pp * (d[0] ** 2 + d[1] ** 2 + d[2] ** 2))
                R = {(0, 0, 0, n): (-2 * pp) ** n * F[n] for n in range(top + 1)}

                def herm(t, u, v, n):
                    if min(t, u, v) < 0:
                        return 0.0
                    key = (t, u, v, n)
                    if key not in R:
                        ax, m = (0, t) if t else (1, u) if u else (2, v)
                        dn = [(t - 1, u, v), (t, u - 1, v), (t, u, v - 1)][ax]
                        val = d[ax] * herm(*dn, n + 1)
                        if m > 1:
                            dn2 = [(t - 2, u, v), (t, u - 2, v), (t, u, v - 2)][ax]
                            val = val + (m - 1) * herm(*dn2, n + 1)
                        R[key] = val
                    return R[key]
                for (t, u, v), w in D.items():
                    V -= (w[sl] * herm(t, u, v, 0)).sum(0)
    return V


def _exact_vne(mol, grid, case):
    nx, ny, nz, h, o = grid.geometry()
    x, y, z = [(torch.arange(n, dtype=torch.float64, device="cuda") + 0.5) * h for n in (nx, ny, nz)]
    src = torch.zeros((nz, ny, nx), dtype=torch.float64, device="cuda")
    for zt, r in zip(mol.types, mol.coords):
        a = r - numpy.array(o)
        d = torch.sqrt(((x - a[0]) ** 2)[None, None, :] + ((y - a[1]) ** 2)[None, :, None]
                       + ((z - a[2]) ** 2)[:, None, None])
        src += torch.where(d < math.sqrt(3.0) * h, float(zt) * torch.exp(-d), 0.0)
    dif, ads = case["diff"], case["adsorb"]

    def sweep(v):
        out = (1.0 - dif * 16.794682450997072 - ads) * v + src
        for i in (-1, 0, 1):
            for j in (-1, 0, 1):
                for k in (-1, 0, 1):
                    n = abs(i) + abs(j) + abs(k)
                    if n:
                        out += dif / math.sqrt(n) * torch.roll(v, (k, j, i), (0, 1, 2))
        for d in range(3):
            out.select(d, 0).zero_()
            out.select(d, -1).zero_()
        return out

    v = torch.zeros_like(src)
    pairs, most = 0, 10.0 * float(nx * ny * nz) ** (1.0 / 3)
    while True:
        t = sweep(v)
        v = sweep(t)
        pairs += 1
        if float((v - t).abs().sum()) / v.numel() <= 1e-9 or pairs > most:
            return v.reshape(-1), pairs


def exact(case, seed):
    kind = case["kind"]
    if kind == "batch":
        mols, grids = _batch_items(case, seed)
        qs = [_exact_density(m, g, 1)[0] for m, g in zip(mols, grids)]
        return {"q": qs, "v": [_exact_fft(q, m, g, "freespace") for q, m, g in zip(qs, mols, grids)]}
    mol, grid, q = _inputs(case, seed)
    if kind == "density":
        q, total = _exact_density(mol, grid, case["subgrid"])
        return {"q": q, "raw_total": total}
    if kind == "jacobi":
        v, m = _exact_jacobi(q, mol, grid, case)
        return {"v": v, "sweeps": None}
    if kind == "fft":
        return _exact_fft(q if case["precision"] == "fp64" else q.float().double(), mol, grid, case["mode"])
    if kind == "gto":
        if case["where"] == "points":
            return _exact_gto(mol, torch.tensor(grid, device="cuda")).cpu().numpy()
        x, y, z = _axes(grid, 0.0)
        Z, Y, X = torch.meshgrid(z, y, x, indexing="ij")
        return _exact_gto(mol, torch.stack([X.reshape(-1), Y.reshape(-1), Z.reshape(-1)], 1))
    v, pairs = _exact_vne(mol, grid, case)
    return {"v": v, "pairs": None}
