"""Performance cases: what a user of the solver has it do on one GPU.

A case is one of four kinds of call, all through the public Python classes:
  solve     CholeskySolverF/D.solve(b, x): one factored system, k right-hand
            sides (k = 0: a one-dimensional b)
  grad      autograd.solve forward and backward: x and the gradients of b and
            of the stored matrix entries
  refactor  refactorize(values) then solve: new values on a known pattern,
            the step of a loop that changes the matrix
  batch     BatchedSolverF/D.solve: independent systems with right-hand-side
            counts of their own
on three families of matrices: mesh (icosphere subdivision, I + lambda (D - W);
keep < 1: the open mesh of the lowest vertices only), grid2 (2D 5-point Laplacian + shift I) and grid3 (3D 7-point Laplacian + shift I).

prepare() makes the inputs (matrix values and right-hand sides differ by
seed) and the factored solver; run() is one call. exact() solves the same
systems by conjugate gradients in FP64 with torch alone.
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

from cholespy_amd import (BatchedSolverD, BatchedSolverF, CholeskySolverD, CholeskySolverF, MatrixType,
                          autograd, workloads)

DEV = torch.device("cuda" if torch.cuda.is_available() else "cpu")
DTYPE = {"f32": torch.float32, "f64": torch.float64}
SOLVER = {"f32": CholeskySolverF, "f64": CholeskySolverD}
BATCHED = {"f32": BatchedSolverF, "f64": BatchedSolverD}


def listed():
    return [
        # A small mesh's positions smoothed inside an interactive loop: launches and latency.
        {"name": "mesh3_k3_f32", "kind": "solve", "mat": "mesh", "level": 3, "k": 3, "dtype": "f32"},
        # A scalar field on a ragged 2D grid (heat, Poisson), b one-dimensional.
        {"name": "grid2_61x47_vec_f64", "kind": "solve", "mat": "grid2", "nx": 61, "ny": 47, "k": 0, "dtype": "f64"},
        # The ordinary inverse-rendering mesh: 10k vertices, 3 coordinates, FP32.
        {"name": "mesh5_k3_f32", "kind": "solve", "mat": "mesh", "level": 5, "k": 3, "dtype": "f32"},
        # The mesh-smoothing headline: 164k vertices, 3 coordinates, in both precisions.
        {"name": "mesh7_k3_f64", "kind": "solve", "mat": "mesh", "level": 7, "k": 3, "dtype": "f64"},
        {"name": "mesh7_k3_f32", "kind": "solve", "mat": "mesh", "level": 7, "k": 3, "dtype": "f32"},
        # The published benchmark: 41k vertices, 128 right-hand sides, FP32.
        {"name": "mesh6_k128_f32", "kind": "solve", "mat": "mesh", "level": 6, "k": 128, "dtype": "f32"},
        # A large ragged 2D grid with an odd number of right-hand sides in FP64.
        {"name": "grid2_511x389_k17_f64", "kind": "solve", "mat": "grid2", "nx": 511, "ny": 389, "k": 17,
         "dtype": "f64"},
        # A 3D volume with a panel of right-hand sides: the largest factor.
        {"name": "grid3_48_k32_f32", "kind": "solve", "mat": "grid3", "m": 48, "k": 32, "dtype": "f32"},
        # An odd-sized 3D volume with a few right-hand sides in FP64.
        {"name": "grid3_33_k5_f64", "kind": "solve", "mat": "grid3", "m": 33, "k": 5, "dtype": "f64"},
        # An optimisation step through the solve: forward, adjoint solve, entry gradients.
        {"name": "mesh6_k3_grad_f32", "kind": "grad", "mat": "mesh", "level": 6, "k": 3, "dtype": "f32"},
        # New matrix values every step (a changing lambda): refactorize, then solve.
        {"name": "mesh6_k3_refactor_f32", "kind": "refactor", "mat": "mesh", "level": 6, "k": 3, "dtype": "f32"},
        # Many independent grids with 1 to 128 right-hand sides each, one call.
        {"name": "batch64_f32", "kind": "batch", "count": 64, "n_min": 1000, "n_max": 20000, "k_max": 128,
         "dtype": "f32", "set": 0},
    ]


def _log_uniform(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.choices(["solve", "grad", "refactor", "batch"], [7, 1, 1, 1])[0]
    dtype = rng.choice(["f32", "f64"])
    if kind == "batch":
        return {"kind": "batch", "count": rng.randint(8, 48), "n_min": 1000,
                "n_max": int(_log_uniform(rng, 2000, 12000)), "k_max": int(_log_uniform(rng, 2, 129)), "dtype": dtype,
                "set": rng.randint(1, 10 ** 6)}
    mat = rng.choice(["mesh", "grid2", "grid3"]) if kind == "solve" else rng.choice(["mesh", "grid2"])
    case = {"kind": kind, "mat": mat}
    top = 1.0 if kind == "solve" else 0.2
    if mat == "mesh":
        case["level"] = rng.randint(3, 7 if kind == "solve" else 6)
        case["keep"] = round(rng.uniform(0.3, 0.99), 3)
    elif mat == "grid2":
        n, r = _log_uniform(rng, 600, 200000 * top), _log_uniform(rng, 0.25, 4.0)
        case["nx"] = max(8, round(math.sqrt(n * r)))
        case["ny"] = max(8, round(n / case["nx"]))
    else:
        case["m"] = round(_log_uniform(rng, 9, 42))
    # The right-hand sides: as many as the largest listed solve does work for.
    most = _factor_entries(_size_case("grid3", m=48)) * 32 / _factor_entries(case)
    case["k"] = rng.choice([0, 1, 3, 3, int(_log_uniform(rng, 1, 129))])
    case["k"] = min(case["k"], max(3, int(most)))
    if kind == "grad" and case["k"] == 0:
        case["k"] = 1
    if kind != "solve":
        case["k"] = min(case["k"], 16)
    case["dtype"] = dtype
    return case


def _size_case(mat, **size):
    return {"mat": mat, **size}


def _rows(case):
    if case["mat"] == "mesh":
        return int((10 * 4 ** case["level"] + 2) * case.get("keep", 1.0))
    return case["nx"] * case["ny"] if case["mat"] == "grid2" else case["m"] ** 3


def _factor_entries(case):
    """Entries of the Cholesky factor under nested dissection: n log n on
    meshes and 2D grids, n^(4/3) on 3D grids (constants of good orderings)."""
    n = _rows(case)
    if case["mat"] == "grid3":
        return 4.8 * n ** (4.0 / 3.0)
    return (2.9 if case["mat"] == "mesh" else 1.5) * n * math.log2(n)


# -- matrices ---------------------------------------------------------------

@functools.lru_cache(maxsize=16)
def _mesh(level, keep=1.0):
    """(n, idx, positions) of the icosphere, or of its vertices that lie lowest (the faces among them)."""
    n, faces, pos = workloads.icosphere(level, with_positions=True)
    if keep < 1.0:
        low = np.zeros(n, dtype=bool)
        low[np.argsort(pos[:, 2], kind="stable")[:int(n * keep)]] = True
        faces = faces[low[faces].all(axis=1)]
        used = np.unique(faces)
        label = np.full(n, -1, dtype=np.int64)
        label[used] = np.arange(len(used))
        n, faces, pos = len(used), label[faces], pos[used]
    _, idx = workloads.mesh_laplacian(n, faces, 1.0)
    return n, idx, pos


@functools.lru_cache(maxsize=4)
def _grid(mat, *size):
    return (workloads.grid2d_laplacian if mat == "grid2" else workloads.grid3d_laplacian)(*size, 0.0)


def _matrix(case, rng):
    """(n, values, idx) in COO. lambda and shift are multiples of 1/16 and
    1/64, so every value and every sum of duplicates is exact in FP32."""
    if case["mat"] == "mesh":
        n, idx, _ = _mesh(case["level"], case.get("keep", 1.0))
        lam = int(rng.integers(96, 352)) / 16.0
        edges = (idx.shape[1] - n) // 2
        return n, np.concatenate([np.full(edges, -lam), np.full(edges, lam), np.ones(n)]), idx
    size = (case["nx"], case["ny"]) if case["mat"] == "grid2" else (case["m"],)
    values, idx = _grid(case["mat"], *size)
    n = _rows(case)
    values = values.copy()
    values[:n] += int(rng.integers(1, 65)) / 64.0   # the diagonal comes first
    return n, values, idx


def _batch(case, seed):
    """[(n, values, idx, k)]: the sizes belong to the case, the shifts to the seed."""
    rng = np.random.default_rng(seed)
    out = []
    for n, values, idx, k in _batch_patterns(case["count"], case["set"], case["n_min"], case["n_max"], case["k_max"]):
        values = values.copy()
        values[:n] = 4.0 + int(rng.integers(1, 65)) / 64.0
        out.append((n, values, idx, k))
    return out


@functools.lru_cache(maxsize=2)
def _batch_patterns(count, which, n_min, n_max, k_max):
    return workloads.batch_systems(count=count, seed=which, n_min=n_min, n_max=n_max, k_max=k_max)


def _rhs(case, n, seed):
    """Vertex positions with noise where the mesh has 3 right-hand sides, normal values elsewhere."""
    g = torch.Generator(device=DEV).manual_seed(int(seed) + 1)
    k = case["k"]
    b = torch.randn((n, k) if k else (n,), generator=g, device=DEV, dtype=torch.float64)
    if case["mat"] == "mesh" and k == 3:
        b = torch.tensor(_mesh(case["level"], case.get("keep", 1.0))[2], device=DEV) + 0.01 * b
    return b.to(DTYPE[case["dtype"]])


# -- the calls ----------------------------------------------------------------

def prepare(case, seed):
    dt = DTYPE[case["dtype"]]
    if case["kind"] == "batch":
        systems = _batch(case, seed)
        ks = [k for *_, k in systems]
        solver = BATCHED[case["dtype"]]([(n, idx[0], idx[1], v, MatrixType.COO) for n, v, idx, _ in systems])
        g = torch.Generator(device=DEV).manual_seed(int(seed) + 1)
        b = torch.randn(sum(n * k for n, _, _, k in systems), generator=g, device=DEV, dtype=dt)
        return {"kind": "batch", "solver": solver, "ks": ks, "b": b, "x": torch.empty_like(b)}
    n, values, idx = _matrix(case, np.random.default_rng(seed))
    ii, jj = torch.tensor(idx[0], device=DEV), torch.tensor(idx[1], device=DEV)
    vals = torch.tensor(values, device=DEV, dtype=dt)
    b = _rhs(case, n, seed)
    st = {"kind": case["kind"], "b": b}
    if case["kind"] == "refactor":
        # Built from other values on the same pattern; the call brings the new ones.
        old = torch.tensor(_matrix(case, np.random.default_rng(seed + 1000003))[1], device=DEV, dtype=dt)
        st.update(solver=SOLVER[case["dtype"]](n, ii, jj, old, MatrixType.COO), values=vals, x=torch.empty_like(b))
        return st
    st["solver"] = SOLVER[case["dtype"]](n, ii, jj, vals, MatrixType.COO)
    if case["kind"] == "grad":
        rows, cols = autograd.coo_indices(n, ii, jj, MatrixType.COO)
        st.update(rows=rows, cols=cols, values=vals.requires_grad_(), b=b.requires_grad_(), gx=_upstream(b, seed))
    else:
        st["x"] = torch.empty_like(b)
    return st


def _upstream(b, seed):
    g = torch.Generator(device=DEV).manual_seed(int(seed) + 2)
    return torch.randn(b.shape, generator=g, device=DEV, dtype=b.dtype)


def run(state):
    kind, solver, b = state["kind"], state["solver"], state["b"]
    if kind == "batch":
        solver.solve(state["ks"], b, state["x"])
        return state["x"]
    if kind == "grad":
        x = autograd.solve(solver, b, state["values"], state["rows"], state["cols"])
        gb, gv = torch.autograd.grad(x, (b, state["values"]), state["gx"])
        return x.detach(), gb, gv
    if kind == "refactor":
        solver.refactorize(state["values"])
    solver.solve(b, state["x"])
    return state["x"]


def work(case):
    """The factor read by each of the two triangular passes, b read and x
    written once; two operations per factor entry, pass and right-hand side."""
    s = 4 if case["dtype"] == "f32" else 8
    if case["kind"] == "batch":
        entries = vec = flops = 0.0
        for n, _, _, k in _batch_patterns(case["count"], case["set"], case["n_min"], case["n_max"], case["k_max"]):
            e = 1.5 * n * math.log2(n)
            entries, vec, flops = entries + e, vec + 2.0 * n * k, flops + 4.0 * e * k
        return {"bytes": s * (2 * entries + vec), "flops": flops}
    n, k, entries = _rows(case), max(1, case["k"]), _factor_entries(case)
    one = {"bytes": s * (2 * entries + 2.0 * n * k), "flops": 4.0 * entries * k}
    if case["kind"] == "grad":   # two solves; lambda and x gathered, indices read, gradient written
        stored = _stored(case)
        return {"bytes": 2 * one["bytes"] + (8 + s) * stored + s * 2.0 * n * k,
                "flops": 2 * one["flops"] + 4.0 * stored * k}
    if case["kind"] == "refactor":   # the values in, the factor out (about 10 n^1.5 operations), the solve
        return {"bytes": one["bytes"] + s * (_stored(case) + entries), "flops": one["flops"] + 10.0 * n ** 1.5}
    return one


def _stored(case):
    return _mesh(case["level"], case.get("keep", 1.0))[1].shape[1] if case["mat"] == "mesh" else 5.0 * _rows(case)


# -- the same in 64 bits with torch alone -------------------------------------

def _lower_symmetric(n, values, idx):
    """The matrix that entries on and below the diagonal stand for, as FP64 CSR (duplicates summed)."""
    i, j, v = torch.tensor(idx[0], device=DEV), torch.tensor(idx[1], device=DEV), torch.tensor(values, device=DEV)
    low = i >= j
    i, j, v = i[low], j[low], v[low]
    off = i != j
    ij = torch.stack([torch.cat([i, j[off]]), torch.cat([j, i[off]])])
    return torch.sparse_coo_tensor(ij, torch.cat([v, v[off]]), (n, n)).coalesce()


def _cg(a, b):
    """A x = b in FP64 for every column: conjugate gradients, restarted twice on the true residual."""
    ij, v = a.indices(), a.values()
    n, k = b.shape
    # Rows padded to one length: a product is a gather and a weighted sum.
    counts = torch.bincount(ij[0], minlength=n)
    ptr = torch.cumsum(counts, 0) - counts
    width = int(counts.max())
    at = torch.arange(ij.shape[1], device=DEV) - ptr[ij[0]]
    cols = torch.zeros((width, n), dtype=torch.int64, device=DEV)
    vals = torch.zeros((width, n, 1), dtype=torch.float64, device=DEV)
    cols[at, ij[0]] = ij[1]
    vals[at, ij[0], 0] = v

    def mul(x):
        y = vals[0] * x[cols[0]]
        for w in range(1, width):
            y += vals[w] * x[cols[w]]
        return y

    x = torch.zeros_like(b)
    for _ in range(3):
        r = b - mul(x)
        d, p = torch.zeros_like(b), r.clone()
        rr = (r * r).sum(0)
        stop = rr * 1e-26
        for it in range(4000):
            q = mul(p)
            alpha = rr / (p * q).sum(0).clamp_min(1e-300)
            d += alpha * p
            r -= alpha * q
            new = (r * r).sum(0)
            p = r + (new / rr.clamp_min(1e-300)) * p
            rr = new
            if it % 16 == 15 and bool((rr <= stop).all()):
                break
        x = x + d
    return x


def exact(case, seed):
    if case["kind"] == "batch":
        st_b = torch.randn(sum(n * k for n, _, _, k in _batch(case, seed)), device=DEV, dtype=DTYPE[case["dtype"]],
                           generator=torch.Generator(device=DEV).manual_seed(int(seed) + 1)).double()
        out, at = [], 0
        for n, v, idx, k in _batch(case, seed):
            out.append(_cg(_lower_symmetric(n, v, idx), st_b[at:at + n * k].view(n, k)).reshape(-1))
            at += n * k
        return torch.cat(out)
    n, values, idx = _matrix(case, np.random.default_rng(seed))
    b = _rhs(case, n, seed)
    a = _lower_symmetric(n, values, idx)
    x = _cg(a, b.double().reshape(n, -1))
    if case["kind"] != "grad":
        return x.reshape(b.shape)
    lam = _cg(a, _upstream(b, seed).double().reshape(n, -1))
    i, j = torch.tensor(idx[0], device=DEV), torch.tensor(idx[1], device=DEV)
    gv = -((lam[i] * x[j]).sum(-1) + (lam[j] * x[i]).sum(-1))
    gv = torch.where(i == j, -(lam[i] * x[i]).sum(-1), torch.where(i > j, gv, torch.zeros_like(gv)))
    return x.reshape(b.shape), lam.reshape(b.shape), gv
