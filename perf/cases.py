"""The work this library is asked to do, as cases that can be timed and compared.

Each case is one pass through the public Python binding (mtl4gpu, and
mtl4gpu_torch for the differentiated solve) on systems of the kinds the library
is used on: discretised operators on 2D and 3D grids with constant and with
strongly varying coefficients, convection-diffusion with all 27 neighbours, and
a triangulated domain whose numbering is no grid.  The matrices are set up here
with numpy alone, so that `exact` depends on nothing but numpy.
"""
import os
import sys
from functools import lru_cache

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "mtl4-mirror_amd"))
import mtl4gpu as g  # noqa: E402


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # the residual and its norm for a small system: one check in a user's own loop, all latency
        dict(name="residual_grid5_64", op="residual", matrix="grid5", nx=64, ny=64, nz=1),
        # the product on the full-size 3D Poisson matrix, the bandwidth-bound end
        dict(name="spmv_poisson7_128", op="spmv", matrix="poisson7", nx=128, ny=128, nz=128),
        # a preconditioner application on a 2D system of odd sides with varying coefficients
        dict(name="apply_ic0_grid5_301x173", op="apply", matrix="grid5", nx=301, ny=173, nz=1, pc="ic0"),
        # the same on the full-size 3D Poisson system
        dict(name="apply_ic0_poisson7_128", op="apply", matrix="poisson7", nx=128, ny=128, nz=128, pc="ic0"),
        # both directions of ILU(0) on the nonsymmetric 27-point system (bicg and qmr need both)
        dict(name="apply_ilu0_conv27_96", op="apply_both", matrix="conv27", nx=96, ny=96, nz=96, pc="ilu0"),
        # ILU(0) on a triangulated domain: rows of differing length, no grid in the numbering
        dict(name="apply_ilu0_mesh_280x230", op="apply", matrix="mesh", nx=280, ny=230, nz=1, pc="ilu0"),
        # a whole small solve, as the reference's own examples run it
        dict(name="cg_ic0_grid5_64", op="solve", matrix="grid5", nx=64, ny=64, nz=1, pc="ic0", method="cg", rtol=1e-10),
        # the headline solve
        dict(name="cg_ic0_poisson7_128", op="solve", matrix="poisson7", nx=128, ny=128, nz=128, pc="ic0", method="cg",
             rtol=1e-8),
        # a nonsymmetric solve on a grid of odd sides
        dict(name="bicgstab_ilu0_conv27_61x53x47", op="solve", matrix="conv27", nx=61, ny=53, nz=47, pc="ilu0",
             method="bicgstab", rtol=1e-10),
        # single precision inside, refined to double: float factors, vectors and products
        dict(name="refined_ilu0_conv27_96", op="refined", matrix="conv27", nx=96, ny=96, nz=96, pc="ilu0", rtol=1e-10),
        # a differentiated solve: assembly, refactorisation and solve forward, adjoint solve and gradient backward
        dict(name="diff_grid5_256", op="diff", matrix="edges", nx=256, ny=256, nz=1, rtol=1e-10),
        # many small systems with several right-hand sides, factorised and solved together
        dict(name="batch_grid5_96x8", op="batch", matrix="grid5", systems=96, lo=32, hi=256, nrhs=8, rtol=1e-8),
    ]


def _log(rng, lo, hi):
    """A whole number between lo and hi, evenly spread over its logarithm."""
    return int(min(hi, max(lo, round(float(lo) * (float(hi) / lo) ** rng.random()))))


def draw(rng):
    """One more case: the same operations over the same kinds of matrix, any sizes in between."""
    op = rng.choice(["residual", "spmv", "apply", "apply", "apply_both", "solve", "solve", "refined", "diff", "batch"])
    if op == "diff":
        return dict(op=op, matrix="edges", nx=_log(rng, 24, 256), ny=_log(rng, 24, 256), nz=1, rtol=1e-10)
    if op == "batch":
        lo = _log(rng, 20, 64)
        return dict(op=op, matrix="grid5", systems=_log(rng, 8, 96), lo=lo, hi=_log(rng, lo + 1, 200),
                    nrhs=rng.choice([1, 2, 4, 8]), rtol=1e-8)
    kind = rng.choice(["grid5", "poisson7", "conv27", "mesh"])
    if op in ("apply_both", "refined"):
        kind = rng.choice(["conv27", "conv27", "grid5", "mesh"])
    if kind == "grid5":
        size = dict(nx=_log(rng, 40, 700), ny=_log(rng, 40, 700), nz=1)
    elif kind == "mesh":
        size = dict(nx=_log(rng, 40, 300), ny=_log(rng, 40, 240), nz=1)
    else:
        top = 128 if kind == "poisson7" else 96
        size = dict(nx=_log(rng, 12, top), ny=_log(rng, 12, top), nz=_log(rng, 12, top))
    case = dict(op=op, matrix=kind, **size)
    if op in ("residual", "spmv"):
        return case
    symmetric = kind != "conv27"
    case["pc"] = rng.choice(["ic0", "ilu0"]) if kind in ("grid5", "poisson7") and op != "apply_both" else "ilu0"
    if op == "solve":
        if kind == "grid5":   # keep the iteration counts of a drawn solve near the listed ones'
            case.update(nx=min(case["nx"], 300), ny=min(case["ny"], 300))
        case["method"] = "cg" if symmetric else "bicgstab"
        case["rtol"] = rng.choice([1e-8, 1e-10])
    if op == "refined":
        if kind == "grid5":
            case.update(nx=min(case["nx"], 200), ny=min(case["ny"], 200))
        case["rtol"] = 1e-10
    return case


# ---------------------------------------------------------------------------
# matrices, with numpy alone
# ---------------------------------------------------------------------------
_STENCIL = {
    "grid5": [(0, -1, 0), (-1, 0, 0), (0, 0, 0), (1, 0, 0), (0, 1, 0)],
    "poisson7": [(0, 0, -1), (0, -1, 0), (-1, 0, 0), (0, 0, 0), (1, 0, 0), (0, 1, 0), (0, 0, 1)],
    "conv27": [(i, j, k) for k in (-1, 0, 1) for j in (-1, 0, 1) for i in (-1, 0, 1)],
}


@lru_cache(maxsize=2)
def _neighbours(kind, nx, ny, nz):
    """Row of each stencil neighbour of each cell (-1: outside); cell (i, j, k) is row i + nx*(j + ny*k)."""
    n = nx * ny * nz
    r = np.arange(n, dtype=np.int64)
    i, j, k = r % nx, r // nx % ny, r // (nx * ny)
    nb = np.empty((n, len(_STENCIL[kind])), np.int64)
    for m, (di, dj, dk) in enumerate(_STENCIL[kind]):
        ok = (i + di >= 0) & (i + di < nx) & (j + dj >= 0) & (j + dj < ny) & (k + dk >= 0) & (k + dk < nz)
        nb[:, m] = np.where(ok, r + di + nx * (dj + ny * dk), -1)
    return nb


def _grid_values(kind, nx, ny, nz, seed):
    """Entries of the operator, one column per stencil neighbour, 0 outside.

    poisson7 has the constants -1 and 6.  The others have a lognormal
    coefficient per cell (harmonic mean between two cells); conv27 adds a
    velocity (1, 0.5, 0.25) at cell Peclet number 0.5.  A boundary face counts
    towards the diagonal (Dirichlet)."""
    sten = _STENCIL[kind]
    nb = _neighbours(kind, nx, ny, nz)
    n, mid = nx * ny * nz, len(sten) // 2
    vals = np.empty((n, len(sten)))
    if kind == "poisson7":
        vals[:] = np.where(nb >= 0, -1.0, 0.0)
        vals[:, mid] = 6.0
        return nb, vals
    kappa = np.exp(np.random.default_rng(seed).standard_normal((nz, ny, nx)))
    padded = np.pad(kappa, 1)                       # 0 outside the domain
    vel = np.array([1.0, 0.5, 0.25]) / np.sqrt(1.3125) * (0.5 if kind == "conv27" else 0.0)
    diag = np.zeros(n)
    for m, d in enumerate(sten):
        if m == mid:
            continue
        kn = padded[1 + d[2]:1 + d[2] + nz, 1 + d[1]:1 + d[1] + ny, 1 + d[0]:1 + d[0] + nx]
        far = d[0] ** 2 + d[1] ** 2 + d[2] ** 2
        w = (2.0 / far) * kappa * kn / (kappa + kn)
        vals[:, m] = (w * (float(vel @ np.array(d)) / np.sqrt(far) - 1.0)).ravel()
        diag += np.where(kn > 0.0, w, kappa / far).ravel()
    vals[:, mid] = diag
    return nb, vals


def _grid_csr(kind, nx, ny, nz, seed):
    nb, vals = _grid_values(kind, nx, ny, nz, seed)
    keep = np.flatnonzero(nb.ravel() >= 0)
    S = np.searchsorted(keep, np.arange(len(nb) + 1) * nb.shape[1])
    return S, nb.ravel()[keep], vals.ravel()[keep]


def _mesh_csr(nx, ny, seed):
    """A piecewise-linear operator on an elliptic domain with a hole: lattice nodes inside it, numbered row by
    row, each lattice square cut along one of its diagonals at random, lognormal edge weights."""
    rng = np.random.default_rng([seed, 17])
    x, y = (np.arange(nx) + 0.5) / nx - 0.5, (np.arange(ny) + 0.5) / ny - 0.5
    rad = (x[None, :] ** 2 + y[:, None] ** 2) * 4.0
    inside = (rad < 1.0) & ((x[None, :] - 0.2) ** 2 + (y[:, None] + 0.1) ** 2 > 0.006)
    num = np.full((ny, nx), -1, np.int64)
    num[inside] = np.arange(int(inside.sum()))
    n = int(inside.sum())
    flip = rng.random((ny - 1, nx - 1)) < 0.5
    ends = [(num[:, :-1].ravel(), num[:, 1:].ravel()), (num[:-1].ravel(), num[1:].ravel()),
            (num[:-1, :-1][flip], num[1:, 1:][flip]), (num[:-1, 1:][~flip], num[1:, :-1][~flip])]
    a, b = np.concatenate([e[0] for e in ends]), np.concatenate([e[1] for e in ends])
    both = (a >= 0) & (b >= 0)
    a, b = a[both], b[both]
    w = np.exp(rng.standard_normal(len(a)))
    diag = np.bincount(a, w, n) + np.bincount(b, w, n) + 0.05
    rows = np.concatenate([a, b, np.arange(n)])
    cols = np.concatenate([b, a, np.arange(n)])
    v = np.concatenate([-w, -w * (1.0 - 0.3 * rng.random(len(w))), diag])
    order = np.lexsort((cols, rows))
    S = np.concatenate([[0], np.cumsum(np.bincount(rows, minlength=n))]).astype(np.int64)
    return S, cols[order], v[order]


def _symmetric_mesh(S, I, V):
    """The mesh operator with its symmetric part, for conjugate gradients."""
    n = len(S) - 1
    rows = np.repeat(np.arange(n), np.diff(S))
    order = np.lexsort((rows, I))
    return S, I, 0.5 * (V + V[order])   # the pattern is symmetric: sorting by column lists the transpose


@lru_cache(maxsize=2)
def _csr(kind, nx, ny, nz, seed, symmetric):
    if kind == "mesh":
        S, I, V = _mesh_csr(nx, ny, seed)
        return _symmetric_mesh(S, I, V) if symmetric else (S, I, V)
    return _grid_csr(kind, nx, ny, nz, seed)


def _matrix(case, seed):
    # the Poisson operator has no coefficients to draw
    s = 0 if case["matrix"] == "poisson7" else seed
    return _csr(case["matrix"], case["nx"], case["ny"], case["nz"], s,
                case.get("method") == "cg" or case["op"] == "refined")


def _times(S, I, V, x):
    return np.add.reduceat(V * x[I], S[:-1])


def _vector(seed, n, stream=0):
    return np.random.default_rng([seed, 99, stream]).uniform(-1.0, 1.0, n)


def _batch_systems(case, seed):
    rng = np.random.default_rng([seed, 5])
    # the sides are part of the case, the coefficients part of the inputs
    sides = np.random.default_rng(7).integers(case["lo"], case["hi"] + 1, case["systems"])
    systems, xs, bs = [], [], []
    for k, side in enumerate(sides):
        S, I, V = _grid_csr("grid5", int(side), int(side), 1, int(rng.integers(1 << 30)))
        x = rng.uniform(-1.0, 1.0, (len(S) - 1, case["nrhs"]))
        systems.append((S, I, V))
        xs.append(x)
        bs.append(np.stack([_times(S, I, V, x[:, q]) for q in range(case["nrhs"])], axis=1))
    return systems, np.concatenate([x.ravel() for x in xs]), np.concatenate([b.ravel() for b in bs])


def _edges_inputs(case, seed):
    """theta, the true solution x and the true adjoint lam of A(theta), A = sum of theta_e (e_i-e_j)(e_i-e_j)^T
    with boundary edges theta_e e_i e_i^T; edge end points as the binding's EdgeSystem numbers them."""
    e = g.edge_laplacian(case["nx"], case["ny"])
    n = case["nx"] * case["ny"]
    theta = np.exp(np.random.default_rng([seed, 3]).standard_normal(e["n_edges"]))
    return e["ei"], e["ej"], theta, _vector(seed, n, 1), _vector(seed, n, 2)


def _edges_times(ei, ej, theta, x):
    inner = ej >= 0
    d = theta * (x[ei] - np.where(inner, x[np.where(inner, ej, 0)], 0.0))
    out = np.bincount(ei, d, len(x))
    return out - np.bincount(ej[inner], d[inner], len(x))


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _new(n):
    return torch.zeros(n, dtype=torch.float64, device="cuda")


_PC = {"ic0": g.PC_IC0, "ilu0": g.PC_ILU0}


def prepare(case, seed):
    op = case["op"]
    st = {"case": dict(case)}
    if op == "diff":
        import mtl4gpu_torch
        ei, ej, theta, x, lam = _edges_inputs(case, seed)
        st["stream"] = torch.cuda.Stream()
        st["solve"] = mtl4gpu_torch.solve
        with torch.cuda.stream(st["stream"]):
            st["system"] = mtl4gpu_torch.EdgeSystem(case["nx"], case["ny"], rtol=case["rtol"])
        st["theta"] = _dev(theta).requires_grad_()
        st["b"] = _dev(_edges_times(ei, ej, theta, x)).requires_grad_()
        st["gx"] = _dev(_edges_times(ei, ej, theta, lam))
    elif op == "batch":
        systems, _, b = _batch_systems(case, seed)
        st["batch"] = g.Batch(systems)
        st["t"] = [_dev(b), _new(len(b))]
    else:
        S, I, V = _matrix(case, seed)
        n = len(S) - 1
        st["A"] = g.Matrix(S, I, V)
        if "pc" in case:
            st["P"] = g.PC(st["A"], _PC[case["pc"]], np.float32 if op == "refined" else np.float64)
        x = _vector(seed, n)
        st["t"] = [_dev(_times(S, I, V, x) if op in ("solve", "refined") else x), _new(n)]
        if op == "residual":
            st["t"].append(_dev(_vector(seed, n, 1)))
        if op == "apply_both":
            st["t"].append(_new(n))
            st["P"].adjoint_solve(g.Vector(tensor=st["t"][0]), g.Vector(tensor=st["t"][2]))
    if "t" in st:
        st["v"] = [g.Vector(tensor=t) for t in st["t"]]
    torch.cuda.synchronize()
    return st


def run(st):
    case = st["case"]
    op = case["op"]
    if op == "spmv":
        g.spmv(st["A"], st["v"][0], st["v"][1])
        return st["t"][1]
    if op == "residual":
        x, r, b = st["v"]
        g.residual(st["A"], x, b, r)
        return [st["t"][1], g.two_norm(r)]
    if op == "apply":
        st["P"].solve(st["v"][0], st["v"][1])
        return st["t"][1]
    if op == "apply_both":
        st["P"].solve(st["v"][0], st["v"][1])
        st["P"].adjoint_solve(st["v"][0], st["v"][2])
        return st["t"][1:]
    if op == "diff":
        with torch.cuda.stream(st["stream"]):
            x = st["solve"](st["theta"], st["b"], st["system"])
            gtheta, gb = torch.autograd.grad(x, (st["theta"], st["b"]), st["gx"])
        return [x.detach(), gtheta, gb]
    b, x = st["v"][:2]
    x.fill(0.0)
    if op == "batch":
        st["batch"].factor_ic0()
        _, _, err = st["batch"].cg_ic0(case["nrhs"], x, b, 20000, case["rtol"])
        if err.any():
            raise RuntimeError("a system did not converge")
        return st["t"][1]
    it, _ = g.make_iteration(20000, case["rtol"], 0.0, g.two_norm(b), history=False)
    if op == "refined":
        code, _ = g.refined_solve(g.METHOD_BICGSTAB, st["A"], x, b, st["P"], it, 1e-4)
    else:
        code = (g.cg if case["method"] == "cg" else g.bicgstab)(st["A"], x, b, st["P"], it)
    if code != 0:
        raise RuntimeError(f"the solve ended with code {code}")
    return st["t"][1]


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _nnz(case):
    if case["matrix"] == "mesh":
        n = int(0.78 * case["nx"] * case["ny"])
        return n, 7 * n
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    n = nx * ny * nz
    if case["matrix"] == "conv27":
        return n, (3 * nx - 2) * (3 * ny - 2) * (3 * nz - 2)
    faces = 2 * ((nx - 1) * ny * nz + nx * (ny - 1) * nz + nx * ny * (nz - 1))
    return n, n + faces


def _solve_rounds(case, n):
    """A plain estimate of the iterations of a solve: they grow with the longest side."""
    side = max(case["nx"], case["ny"], case["nz"])
    if case["matrix"] == "conv27":
        return 0.4 * side * (1.3 if case["op"] == "refined" else 1.0)
    per = {"poisson7": 0.8, "grid5": 1.25, "edges": 1.65, "mesh": 1.3}[case["matrix"]]
    return per * side * (1.25 if case["rtol"] < 1e-9 else 1.0)


def work(case):
    op = case["op"]
    if op == "batch":
        sides = np.random.default_rng(7).integers(case["lo"], case["hi"] + 1, case["systems"]).astype(float)
        rounds = 1.25 * sides
        # per right-hand side and iteration: x, r, p, q, z once each way; the matrix and the factor once per system
        each = sides ** 2 * (case["nrhs"] * 10 * 8 + 5 * 12 + 2 * 3 * 12)
        return {"bytes": float((each * rounds).sum()), "flops": float((sides ** 2 * rounds).sum() * case["nrhs"] * 34)}
    if op == "diff":
        n, nnz = _nnz(dict(case, matrix="grid5"))
        per = 12 * nnz + 12 * (nnz + n) + 8 * 18 * n
        rounds = 2 * _solve_rounds(case, n)
        return {"bytes": rounds * per, "flops": rounds * (4 * nnz + 14 * n)}
    n, nnz = _nnz(case)
    product = 12 * nnz + 4 * (n + 1) + 16 * n
    entries = nnz if case.get("pc") == "ilu0" else nnz + n   # ic_0 reads its factor once for each sweep
    apply = 12 * entries + 8 * (n + 1) + 16 * n
    if op == "spmv":
        return {"bytes": product, "flops": 2 * nnz}
    if op == "residual":
        return {"bytes": product + 8 * n, "flops": 2 * nnz + 3 * n}
    if op == "apply":
        return {"bytes": apply, "flops": 2 * entries}
    if op == "apply_both":
        return {"bytes": 2 * apply, "flops": 4 * entries}
    rounds = _solve_rounds(case, n)
    if op == "solve" and case["method"] == "cg":
        return {"bytes": rounds * (product + apply + 72 * n), "flops": rounds * (2 * nnz + 2 * entries + 10 * n)}
    half = 0.5 if op == "refined" else 1.0
    return {"bytes": rounds * half * 2 * (product + apply + 72 * n), "flops": rounds * 2 * (2 * nnz + 2 * entries + 12 * n)}


# ---------------------------------------------------------------------------
# what the results are, from numpy in double precision
# ---------------------------------------------------------------------------
def _grid_ilu0(kind, nx, ny, nz, vals):
    """ILU(0) without fill on a grid stencil, cell by cell along the planes i + 2j + 4k, which no stencil entry
    joins to itself.  (On 5 and 7 points this is also the incomplete Cholesky factorisation.)  Returns the
    planes, the neighbours (n: outside, with a row of zeros) and the factors, diagonal inverted."""
    sten, n = _STENCIL[kind], nx * ny * nz
    mid, where = len(sten) // 2, {d: m for m, d in enumerate(sten)}
    nb = np.where(_neighbours(kind, nx, ny, nz) >= 0, _neighbours(kind, nx, ny, nz), n)
    r = np.arange(n)
    t = r % nx + 2 * (r // nx % ny) + 4 * (r // (nx * ny))
    order = np.argsort(t, kind="stable")
    planes = np.split(order, np.flatnonzero(np.diff(t[order])) + 1)
    f = np.concatenate([vals, np.zeros((1, len(sten)))])
    for rows in planes:
        v = f[rows]
        for p in range(mid):
            k = nb[rows, p]
            v[:, p] *= f[k, mid]
            for q in range(mid + 1, len(sten)):
                s = where.get(tuple(a + b for a, b in zip(sten[p], sten[q])))
                if s is not None:
                    v[:, s] -= v[:, p] * f[k, q]
        v[:, mid] = 1.0 / v[:, mid]
        f[rows] = v
    return planes, nb, f


def _grid_apply(kind, planes, nb, f, x, adjoint=False):
    n, m = len(x), f.shape[1]
    mid = m // 2
    y = np.concatenate([x, [0.0]])
    for rows in planes:
        acc = y[rows]
        for p in range(mid):
            k = nb[rows, p]
            acc = acc - (f[k, m - 1 - p] if adjoint else f[rows, p]) * y[k]
        y[rows] = acc * f[rows, mid] if adjoint else acc
    for rows in reversed(planes):
        acc = y[rows]
        for p in range(mid + 1, m):
            k = nb[rows, p]
            acc = acc - (f[k, m - 1 - p] if adjoint else f[rows, p]) * y[k]
        y[rows] = acc if adjoint else acc * f[rows, mid]
    return y[:n]


def _general_apply(S, I, V, x, adjoint=False):
    """ILU(0) and its two triangular solves, row by row."""
    n = len(S) - 1
    rows = [dict(zip(I[S[r]:S[r + 1]].tolist(), V[S[r]:S[r + 1]].tolist())) for r in range(n)]
    for r in range(n):
        row = rows[r]
        for k in sorted(c for c in row if c < r):
            up = rows[k]
            row[k] = l = row[k] / up[k]
            for c, u in up.items():
                if c > k and c in row:
                    row[c] -= l * u
    y = x.tolist()
    if adjoint:
        for r in range(n):
            y[r] /= rows[r][r]
            for c, u in rows[r].items():
                if c > r:
                    y[c] -= u * y[r]
        for r in range(n - 1, -1, -1):
            for c, l in rows[r].items():
                if c < r:
                    y[c] -= l * y[r]
    else:
        for r in range(n):
            y[r] -= sum(l * y[c] for c, l in rows[r].items() if c < r)
        for r in range(n - 1, -1, -1):
            y[r] = (y[r] - sum(u * y[c] for c, u in rows[r].items() if c > r)) / rows[r][r]
    return np.array(y)


def exact(case, seed):
    op = case["op"]
    if op == "batch":
        return _batch_systems(case, seed)[1]      # b is A times this x
    if op == "diff":
        ei, ej, theta, x, lam = _edges_inputs(case, seed)
        inner = ej >= 0
        far = np.where(inner, ej, 0)
        grad = -(lam[ei] - np.where(inner, lam[far], 0.0)) * (x[ei] - np.where(inner, x[far], 0.0))
        return [x, grad, lam]
    S, I, V = _matrix(case, seed)
    x = _vector(seed, len(S) - 1)
    if op in ("solve", "refined"):
        return x                                  # b is A times this x
    if op == "spmv":
        return _times(S, I, V, x)
    if op == "residual":
        r = _vector(seed, len(x), 1) - _times(S, I, V, x)
        return [r, float(np.sqrt(r @ r))]
    if case["matrix"] == "mesh":
        if case.get("pc") == "ic0":
            return None
        out = [_general_apply(S, I, V, x, adj) for adj in ((False, True) if op == "apply_both" else (False,))]
    else:
        shape = case["matrix"], case["nx"], case["ny"], case["nz"]
        nb, vals = _grid_values(*shape, 0 if case["matrix"] == "poisson7" else seed)
        planes, nb, f = _grid_ilu0(*shape, vals)
        out = [_grid_apply(case["matrix"], planes, nb, f, x, adj)
               for adj in ((False, True) if op == "apply_both" else (False,))]
    return out if op == "apply_both" else out[0]
