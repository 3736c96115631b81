"""Ill-conditioned systems keep a small residual in solves with a dense top:
whole systems and tops between the passes, kappa about 1e4 and 1e6, b = A x.

Tolerance: each of the solve's products rounds X, its input and its result,
and A's entries are at most its norm, so ||b - A x|| is a few units of rounding
of ||A|| ||x||, about ||b||: at most 16 (u = 2^-24, 2^-53). A product with a
rounded inverse of A, whose residual is kappa u, is 100 to 10,000 times off."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from cholespy_amd import CholeskySolverD, CholeskySolverF, MatrixType, workloads

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda")
UNIT = {np.float32: 2.0 ** -24, np.float64: 2.0 ** -53}


def _systems():
    for level in (3, 4, 5):
        n, faces = workloads.icosphere(level)
        for lam in (1e3, 1e5):   # kappa ~ 10 lambda
            yield f"ico{level}-{lam:g}", n, *workloads.mesh_laplacian(n, faces, lam)
    for shift in (1e-3, 1e-5):   # Neumann: kappa = 12 / shift
        yield f"cube16-{shift:g}", 16 ** 3, *workloads.grid3d_laplacian(16, shift)
        yield f"cube24-{shift:g}", 24 ** 3, *workloads.grid3d_laplacian(24, shift)


SYSTEMS = list(_systems())


@pytest.mark.parametrize("name,n,values,idx", SYSTEMS, ids=[s[0] for s in SYSTEMS])
@pytest.mark.parametrize("cls,dtype", [(CholeskySolverF, np.float32), (CholeskySolverD, np.float64)])
def test_residual(name, n, values, idx, cls, dtype):
    ext = np.longdouble
    v = values.astype(dtype)
    s = cls(n, *(torch.tensor(a, device=DEV) for a in (idx[0], idx[1], v)), MatrixType.COO)
    assert (s._plan_arrays()["fwd_task"][:, 3] == 4).any()
    # A from the entries on and below the diagonal (duplicates added), in extended precision.
    low = idx[0] >= idx[1]
    i, j, a = idx[0][low], idx[1][low], v[low].astype(ext)
    off = i != j
    i, j, a = np.concatenate([i, j[off]]), np.concatenate([j, i[off]]), np.concatenate([a, a[off]])
    order = np.argsort(i, kind="stable")
    i, j, a = i[order], j[order], a[order]
    first = np.flatnonzero(np.r_[True, i[1:] != i[:-1]])

    def times(x):
        return np.add.reduceat(a[:, None] * x[j], first, axis=0)

    for k in (1, 3, 16, 33):
        x = np.random.default_rng(k).standard_normal((n, k))
        b = times(x.astype(ext)).astype(dtype)
        bt = torch.tensor(b, device=DEV)
        xt = torch.zeros_like(bt)
        s.solve(bt, xt)
        torch.cuda.synchronize()
        s._check()
        r = (b.astype(ext) - times(xt.cpu().numpy().astype(ext))).astype(np.float64)
        res = (np.linalg.norm(r, axis=0) / np.linalg.norm(b.astype(np.float64), axis=0)).max()
        print(name, dtype.__name__, k, res / UNIT[dtype])
        assert res <= 16 * UNIT[dtype], (name, k, res)
