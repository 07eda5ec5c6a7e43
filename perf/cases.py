"""The work that users of this package have it do, as cases to time: solves, preconditioner
applications, batches, the differentiable solve and the reference's one-shot call, over the
sizes that the repository's workloads, tests and benchmark use.

A case names its `kind` (the entry point), the grid, the field of conductivities ("laplace" or
"varcoef"), the order inside the nested-dissection blocks ("mis", "static" or "natural"), the
leaves and the precision of the factor.  Every vector is drawn from the seed; the matrix and its
factor are those of the grid (a program factors once and solves for many right-hand sides), except
for the kinds "grad" and "oneshot", whose weights are drawn from the seed too.

Solves return the solution alone: the iteration count and the residual norm that come with it say
where a tolerance was crossed and move with the last bit of every sum.
"""
import functools
import json
import math

import numpy as np
import torch

import rchol_amd
from rchol_amd import autograd as AG
from rchol_amd import factor as F

TOL = 1e-10    # the tolerance of the repository's benchmark and configurations
MAXIT = 5000


def listed():
    return [
        # the benchmark's headline problem, FP32 factor: the largest solve
        {"name": "pcg-mixed-256", "kind": "pcg", "field": "varcoef", "nx": 256, "ny": 256,
         "nz": 256, "order": "mis", "leaves": 128, "prec": "fp32", "perm": False},
        # the 128^3 Laplacian of 64 leaves in FP64: an ordinary solve
        {"name": "pcg-fp64-128", "kind": "pcg", "field": "laplace", "nx": 128, "ny": 128,
         "nz": 128, "order": "mis", "leaves": 64, "prec": "fp64", "perm": False},
        # an odd box with vectors in the caller's numbering (the engine permutes)
        {"name": "pcg-mixed-odd", "kind": "pcg", "field": "varcoef", "nx": 97, "ny": 61,
         "nz": 83, "order": "mis", "leaves": 16, "prec": "fp32", "perm": True},
        # a small solve: latency and launches
        {"name": "pcg-fp64-32", "kind": "pcg", "field": "varcoef", "nx": 32, "ny": 32,
         "nz": 32, "order": "mis", "leaves": 8, "prec": "fp64", "perm": False},
        # a factor in the reference's own order (natural inside the blocks), used as it is
        {"name": "pcg-static-64", "kind": "pcg", "field": "laplace", "nx": 64, "ny": 64,
         "nz": 64, "order": "static", "leaves": 16, "prec": "fp64", "perm": False},
        # the reference's sequential example: natural order, no dissection
        {"name": "pcg-natural-24", "kind": "pcg", "field": "laplace", "nx": 24, "ny": 24,
         "nz": 24, "order": "natural", "leaves": 1, "prec": "fp64", "perm": False},
        # one application inside a caller's own Krylov loop
        {"name": "precond-fp64-128", "kind": "precond", "field": "varcoef", "nx": 128, "ny": 128,
         "nz": 128, "order": "mis", "leaves": 64, "prec": "fp64", "perm": False},
        # the smallest call
        {"name": "precond-fp64-20", "kind": "precond", "field": "laplace", "nx": 20, "ny": 20,
         "nz": 20, "order": "mis", "leaves": 4, "prec": "fp64", "perm": False},
        # a full block of right-hand sides on one matrix, FP32 factor
        {"name": "batch32-mixed-100", "kind": "batch", "field": "varcoef", "nx": 100, "ny": 100,
         "nz": 100, "order": "mis", "leaves": 16, "prec": "fp32", "k": 32},
        # many uneven two-dimensional systems, solved together from host arrays
        {"name": "uneven-24", "kind": "segments", "nsys": 24, "lo": 64, "hi": 512,
         "prec": "fp32"},
        # forward and adjoint of the differentiable solve, factor of the weights in hand
        {"name": "grad-64", "kind": "grad", "nx": 64, "ny": 64, "nz": 64, "leaves": 16,
         "prec": "fp32"},
        # the reference's Python call on host arrays: upload, solve, release
        {"name": "oneshot-40", "kind": "oneshot", "nx": 40, "ny": 40, "nz": 40, "leaves": 8},
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _box(rng, lo, hi):
    """Three extents about one side drawn over the logarithm of [lo, hi]."""
    s = _logint(rng, lo, hi)
    return [max(4, min(hi, int(round(s * rng.uniform(0.8, 1.2))))) for _ in range(3)]


def _leaves(rng, n):
    """A power of two: blocks of about 4,000 rows up to a few times more, at most 128."""
    most = max(1, min(7, int(math.log2(max(2, n / 4096)))))
    return 2 ** max(1, most - rng.randrange(2))


def draw(rng):
    kind = rng.choice(["pcg", "pcg", "pcg", "deep", "precond", "precond", "batch", "segments",
                       "grad", "oneshot"])
    prec = rng.choice(["fp32", "fp64"])
    if kind == "pcg":
        nx, ny, nz = _box(rng, 14, 210)
        return {"kind": "pcg", "field": rng.choice(["laplace", "varcoef"]), "nx": nx, "ny": ny,
                "nz": nz, "order": "mis", "leaves": _leaves(rng, nx * ny * nz), "prec": prec,
                "perm": rng.random() < 0.5}
    if kind == "deep":
        nx, ny, nz = _box(rng, 14, 72)
        return {"kind": "pcg", "field": rng.choice(["laplace", "varcoef"]), "nx": nx, "ny": ny,
                "nz": nz, "order": "static", "leaves": _leaves(rng, nx * ny * nz), "prec": prec,
                "perm": rng.random() < 0.5}
    if kind == "precond":
        nx, ny, nz = _box(rng, 10, 160)
        return {"kind": "precond", "field": rng.choice(["laplace", "varcoef"]), "nx": nx,
                "ny": ny, "nz": nz, "order": "mis", "leaves": _leaves(rng, nx * ny * nz),
                "prec": "fp64", "perm": rng.random() < 0.5}
    if kind == "batch":
        nx, ny, nz = _box(rng, 14, 100)
        return {"kind": "batch", "field": rng.choice(["laplace", "varcoef"]), "nx": nx, "ny": ny,
                "nz": nz, "order": "mis", "leaves": _leaves(rng, nx * ny * nz), "prec": prec,
                "k": rng.choice([4, 8, 16, 32])}
    if kind == "segments":
        lo = _logint(rng, 16, 96)
        return {"kind": "segments", "nsys": _logint(rng, 3, 32), "lo": lo,
                "hi": _logint(rng, 2 * lo, 512), "prec": prec}
    nx, ny, nz = _box(rng, 12, 72 if kind == "grad" else 48)
    c = {"kind": kind, "nx": nx, "ny": ny, "nz": nz, "leaves": _leaves(rng, nx * ny * nz)}
    if kind == "grad":
        c["prec"] = prec
    return c


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------
def _prec(case):
    return rchol_amd.FP32 if case.get("prec") == "fp32" else rchol_amd.FP64


def _depth(leaves):
    return int(math.log2(leaves)) + 1


def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


@functools.lru_cache(maxsize=2)
def _system_of(key):
    """(A(perm, perm), stored factor, perm) of a grid case."""
    c = json.loads(key)
    dims = (c["nx"], c["ny"], c["nz"])
    if c["field"] == "laplace" and len(set(dims)) == 1:
        A = F.laplace_3d(dims[0])
    elif c["field"] == "laplace":
        # unit conductivities on a box: the grid Laplacian with a small shift
        A = F.grid_laplacian(*dims, np.ones(F.grid_edges(*dims)[0].size), 1e-2)
    else:
        A = F.varcoef_3d(*dims, 1.5, 1e-3, 20261202)
    if c["order"] == "natural":
        Gs, po, _ = F.factor(A, None, [A.shape[0]], "static", 1)
        return A, Gs, po
    perm, blocks = F.nd_grid(*dims, _depth(c["leaves"]))
    Gs, po, _ = F.factor(A, perm, blocks, c["order"], 1)
    return F.permute(A, po), Gs, po


def _system(case):
    return _system_of(json.dumps({k: case[k] for k in ("field", "nx", "ny", "nz", "order",
                                                       "leaves")}))


@functools.lru_cache(maxsize=2)
def _stack_of(nsys, lo, hi):
    """Block-diagonal stack of nsys 2D systems, sides log-uniform in [lo, hi]."""
    rng = np.random.default_rng(48)
    sides = np.exp(rng.uniform(np.log(lo), np.log(hi), nsys)).astype(int)
    systems = []
    for i, s in enumerate(sides):
        s = int(s)
        A = F.varcoef_3d(s, s, 1, 1.0, 0.0, 1000 + i)
        perm, blocks = F.nd_grid(s, s, 1, _depth(8 if s >= 32 else 2))
        Gs, po, _ = F.factor(A, perm, blocks, "mis", i + 1)
        systems.append((F.permute(A, po), Gs))
    return rchol_amd.stack_systems(systems)


def _rhs(n, seed, k=None):
    """b ~ U[-1, 1] (n, or n x k), from the seed."""
    return np.random.default_rng(seed).uniform(-1.0, 1.0, n if k is None else (n, k))


def _weights(case, seed):
    """Edge parameters, right-hand side and target of a training step."""
    m = F.grid_edges(case["nx"], case["ny"], case["nz"])[0].size
    n = case["nx"] * case["ny"] * case["nz"]
    rng = np.random.default_rng(seed)
    return (np.logaddexp(0.0, rng.standard_normal(m)), rng.uniform(-1.0, 1.0, n),
            rng.uniform(-1.0, 1.0, n))


def _oneshot_inputs(case, seed):
    """A(perm, perm) of random weights, its factor as scipy G and G^T, and b."""
    w, b, _ = _weights(case, seed)
    dims = (case["nx"], case["ny"], case["nz"])
    A = F.grid_laplacian(*dims, w, 1e-2)
    perm, blocks = F.nd_grid(*dims, _depth(case["leaves"]))
    Gs, po, _ = F.factor(A, perm, blocks, "mis", 1)
    G = F.lower(Gs)
    return F.permute(A, po), b, G, G.T.tocsr()


def prepare(case, seed):
    kind = case["kind"]
    dev = _device()
    if kind in ("pcg", "precond", "batch"):
        A, Gs, po = _system(case)
        s = rchol_amd.Solver(A, Gs, _prec(case))
        if case.get("perm"):
            s.set_perm(po)
        b = torch.as_tensor(_rhs(A.shape[0], seed, case.get("k")), device=dev)
        return {"kind": kind, "solver": s, "b": b, "x": torch.empty_like(b), "k": case.get("k")}
    if kind == "segments":
        A, G, off = _stack_of(case["nsys"], case["lo"], case["hi"])
        s = rchol_amd.Solver(A, G, _prec(case))
        s.set_segments(off)
        return {"kind": kind, "solver": s, "b": _rhs(A.shape[0], seed)}
    if kind == "grad":
        w, b, t = _weights(case, seed)
        prob = AG.GridLaplacian(case["nx"], case["ny"], case["nz"], shift=1e-2,
                                leaves=case["leaves"], precision=_prec(case), tol=TOL)
        w = torch.as_tensor(w, device=dev).requires_grad_()
        prob.solver_for(w.detach())
        return {"kind": kind, "prob": prob, "w": w,
                "b": torch.as_tensor(b, device=dev).requires_grad_(),
                "t": torch.as_tensor(t, device=dev)}
    A, b, G, Gt = _oneshot_inputs(case, seed)
    return {"kind": kind, "A": A, "b": b, "G": G, "Gt": Gt}


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------
def run(state):
    kind = state["kind"]
    if kind == "pcg":
        state["solver"].pcg_device(state["b"].data_ptr(), state["x"].data_ptr(), TOL, MAXIT)
        return state["x"]
    if kind == "precond":
        state["solver"].precond_device(state["b"].data_ptr(), state["x"].data_ptr())
        return state["x"]
    if kind == "batch":
        state["solver"].pcg_batch_device(state["k"], state["b"].data_ptr(),
                                         state["x"].data_ptr(), TOL, MAXIT)
        return state["x"]
    if kind == "segments":
        return state["solver"].pcg_segments(state["b"], TOL, MAXIT)[0]
    if kind == "grad":
        w, b = state["w"], state["b"]
        w.grad = b.grad = None
        x = AG.solve(w, b, state["prob"])
        ((x - state["t"]) ** 2).sum().backward()
        return {"x": x.detach(), "gw": w.grad, "gb": b.grad}
    return rchol_amd.pcg(state["A"], state["b"], TOL, MAXIT, state["G"], state["Gt"])[0]


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------
def _pcg_bytes(n, nnz_a, nnz_g, prec, its, k=1):
    """One solve of k columns: per iteration both sweeps, A p and the vector updates, each
    matrix entry read once for all columns, each vector read or written once per stage."""
    s = 4 if prec == "fp32" else 8
    sweeps = 2 * (nnz_g * (s + 4) + 4 * n) + k * n * (8 + 3 * s)
    spmv = 12 * nnz_a + 4 * n + k * n * (s + 40)
    update = 48 * n * k
    return its * (sweeps + spmv + update) + k * n * 16


def _its(n, order="mis"):
    """Iterations to 1e-10 that these factors take (25 at 32^3 to 39 at 256^3)."""
    return int(round(5 + (4.2 if order == "mis" else 3.4) * math.log2(n) / 3))


def work(case):
    kind = case["kind"]
    prec = case.get("prec", "fp64")
    if kind == "segments":
        A, G, _ = _stack_of(case["nsys"], case["lo"], case["hi"])
        n, nnz_a, nnz_g, its = A.shape[0], A.nnz, int(G[0][-1]), 30
    else:
        n = case["nx"] * case["ny"] * case["nz"]
        nnz_a = 7 * n
        # entries of a factor with its diagonal: 1.3 to 1.9 times A's lower half
        nnz_g = int((9.7 if case.get("order", "mis") == "mis" else 13.5) * n)
        its = _its(n, case.get("order", "mis"))
    if kind == "precond":
        s = 4 if prec == "fp32" else 8
        return {"bytes": 2 * (nnz_g * (s + 4) + 4 * n) + n * (16 + 2 * s),
                "flops": 4 * nnz_g}
    k = case.get("k", 1)
    nbytes = _pcg_bytes(n, nnz_a, nnz_g, prec, its, k)
    flops = its * k * (4 * nnz_g + 2 * nnz_a + 12 * n)
    if kind == "grad":
        m = 3 * n
        return {"bytes": 2 * nbytes + 24 * m + 40 * n, "flops": 2 * flops}
    return {"bytes": nbytes, "flops": flops}


# ---------------------------------------------------------------------------
# The same in 64 bits, by torch alone
# ---------------------------------------------------------------------------
def _csr(A):
    dev = _device()
    return torch.sparse_csr_tensor(torch.as_tensor(A.indptr.astype(np.int64), device=dev),
                                   torch.as_tensor(A.indices.astype(np.int64), device=dev),
                                   torch.as_tensor(np.array(A.data), device=dev), size=A.shape)


def _cg(A, d, b):
    """A^-1 b (b: n x k) by Jacobi-preconditioned CG, restarted on the true residual."""
    x = torch.zeros_like(b)
    nb = b.norm(dim=0).clamp_min(1e-300)
    for _ in range(3):
        r = b - A @ x
        z = r / d
        p = z.clone()
        rz = (r * z).sum(dim=0)
        start = r.norm(dim=0).clamp_min(1e-300)
        goal = torch.maximum(1e-15 * nb, 1e-13 * start)
        for it in range(20000):
            q = A @ p
            al = rz / (p * q).sum(dim=0).clamp_min(1e-300)
            x = x + al * p
            r = r - al * q
            if it % 25 == 24 and bool((r.norm(dim=0) <= goal).all()):
                break
            z = r / d
            new = (r * z).sum(dim=0)
            p = z + (new / rz.clamp_min(1e-300)) * p
            rz = new
    return x


def _solve(A, b):
    dev = _device()
    bt = torch.as_tensor(b, device=dev).reshape(A.shape[0], -1)
    d = torch.as_tensor(A.diagonal(), device=dev).reshape(-1, 1)
    return _cg(_csr(A), d, bt).reshape(np.shape(b))


def _sweep(T, d, b):
    """T^-1 b for a triangular T = diag(d) + (T - diag(d)), by substituting until nothing
    changes: at most as many times as T has dependency levels."""
    x = b / d
    for _ in range(20000):
        y = (b - T @ x) / d
        if bool((y - x).abs().max() <= 1e-17 * y.abs().max()):
            return y
        x = y
    return x


def _triangles(Gs):
    """Strict G, strict G^T (both CSR) and the diagonal of a stored factor."""
    dev = _device()
    cp = torch.as_tensor(np.asarray(Gs[0]).astype(np.int64), device=dev)
    ri = torch.as_tensor(np.asarray(Gs[1]).astype(np.int64), device=dev)
    v = torch.as_tensor(np.array(Gs[2]), device=dev)
    n = cp.numel() - 1
    col = torch.repeat_interleave(torch.arange(n, device=dev), cp[1:] - cp[:-1])
    on = ri == col
    d = torch.zeros(n, dtype=v.dtype, device=dev)
    d[col[on]] = v[on]
    r, c, w = ri[~on], col[~on], v[~on]

    def csr(rows, cols):
        order = torch.argsort(rows * n + cols)
        ptr = torch.zeros(n + 1, dtype=torch.int64, device=dev)
        ptr[1:] = torch.bincount(rows, minlength=n).cumsum(0)
        return torch.sparse_csr_tensor(ptr, cols[order], w[order], size=(n, n))

    return csr(r, c), csr(c, r), d


def exact(case, seed):
    kind = case["kind"]
    if kind == "segments":
        A, _, _ = _stack_of(case["nsys"], case["lo"], case["hi"])
        if A.shape[0] > 2_000_000:
            return None
        return _solve(A, _rhs(A.shape[0], seed)).cpu().numpy()
    n = case["nx"] * case["ny"] * case["nz"]
    if n > 2_500_000:
        return None  # the factor and the reference solve together take too long
    if kind == "oneshot":
        A, b, _, _ = _oneshot_inputs(case, seed)
        return _solve(A, b).cpu().numpy()
    if kind == "grad":
        w, b, t = _weights(case, seed)
        dims = (case["nx"], case["ny"], case["nz"])
        A = F.grid_laplacian(*dims, w, 1e-2)
        u, v = F.grid_edges(*dims)
        x = _solve(A, b).cpu().numpy()
        lam = _solve(A, 2.0 * (x - t)).cpu().numpy()
        return {"x": x, "gw": -(lam[u] - lam[v]) * (x[u] - x[v]), "gb": lam}
    A, Gs, po = _system(case)
    b = _rhs(n, seed, case.get("k"))
    p = po.astype(np.int64)
    bp = b[p] if case.get("perm") else b
    if kind == "precond":
        L, U, d = _triangles(Gs)
        xp = _sweep(U, d, _sweep(L, d, torch.as_tensor(bp, device=_device())))
    else:
        xp = _solve(A, bp)
    if not case.get("perm"):
        return xp
    x = torch.empty_like(xp)
    x[torch.as_tensor(p, device=xp.device)] = xp
    return x
