"""Systems of several unconnected parts with a dense top: a NaN or an infinity
in one part's right-hand side leaves the solutions of the others bit for bit
as they were, and each part matches the oracle (kappa < 20: the tolerances of
the other parity tests). Parts of one row, parts that end inside a panel of 16
rows, systems of top rows only and systems with levels below the top."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from cholespy_amd import CholeskySolverD, CholeskySolverF, MatrixType, workloads
from oracle import oracle

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda")
TOL = {np.float32: 2e-5, np.float64: 1e-12}


@pytest.mark.parametrize("grids", [[(30, 31), (3, 3), (1, 1), (40, 17), (25, 25)], [(16, 16)] * 9, [(1, 1)] * 40,
                                   [(101, 97), (61, 47), (5, 1), (89, 83)]], ids=["small", "equal", "dust", "large"])
@pytest.mark.parametrize("cls,dtype", [(CholeskySolverF, np.float32), (CholeskySolverD, np.float64)])
def test_parts_stay_apart(grids, cls, dtype):
    n, values, rows, cols, part = 0, [], [], [], []
    for g, (nx, ny) in enumerate(grids):
        v, idx = workloads.grid2d_laplacian(nx, ny, 0.5)
        values.append(v)
        rows.append(idx[0] + n)
        cols.append(idx[1] + n)
        part.append(np.full(nx * ny, g))
        n += nx * ny
    part = np.concatenate(part)
    s = cls(n, *(torch.tensor(np.concatenate(a), device=DEV) for a in (rows, cols, values)), MatrixType.COO)
    if grids != [(1, 1)] * 40:
        assert (s._plan_arrays()["fwd_task"][:, 3] == 4).any()
    for k in (1, 3, 7, 20, 50):
        b = np.random.default_rng(k).standard_normal((n, k)).astype(dtype)

        def solve(b):
            bt = torch.tensor(b, device=DEV)
            xt = torch.zeros_like(bt)
            s.solve(bt, xt)
            torch.cuda.synchronize()
            s._check()
            return xt.cpu().numpy()

        x = solve(b)
        ref = oracle.solve(s._factor(), b, dtype)
        assert np.abs(x - ref).max() / np.abs(ref).max() < TOL[dtype], k
        for bad in (np.nan, np.inf):
            for g in (0, len(grids) - 1):
                bb = b.copy()
                bb[np.flatnonzero(part == g)[0], 0] = bad
                xb = solve(bb)
                assert np.array_equal(xb[part != g], x[part != g]), (k, bad, g)
                assert not np.isfinite(xb[part == g, 0]).any() and np.array_equal(xb[:, 1:], x[:, 1:]), (k, bad, g)
