"""FP64 leaf units (one wavefront a leaf task at more than 16 right-hand sides)
are as accurate as the workgroup tasks they replace: the error against the
solution in extended precision is at most 4 % above theirs. (Both round each
product once; only the order of the sums differs, and over 14,000 rows and 20
columns chance moves the ratio by about 1 %.)"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from cholespy_amd import CholeskySolverD, MatrixType, workloads
from oracle import oracle

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda")


@pytest.mark.parametrize("system", ["grid2", "grid3"])
def test_error_of_leaf_units(system, monkeypatch):
    monkeypatch.setenv("CHOLESPY_DENSE_TOP", "0")
    if system == "grid2":
        n, (v, idx) = 151 * 97, workloads.grid2d_laplacian(151, 97, 0.25)
    else:
        n, (v, idx) = 21 ** 3, workloads.grid3d_laplacian(21, 0.25)
    ext = np.longdouble
    low = idx[0] >= idx[1]
    i, j, a = idx[0][low], idx[1][low], v[low].astype(ext)
    off = i != j
    i, j, a = np.concatenate([i, j[off]]), np.concatenate([j, i[off]]), np.concatenate([a, a[off]])
    order = np.argsort(i, kind="stable")
    i, j, a = i[order], j[order], a[order]
    first = np.flatnonzero(np.r_[True, i[1:] != i[:-1]])
    b = np.random.default_rng(1).standard_normal((n, 20))
    errors = {}
    for leaves in ("1", "0"):
        monkeypatch.setenv("CHOLESPY_LEAF_KERNELS", leaves)
        s = CholeskySolverD(n, *(torch.tensor(q, device=DEV) for q in (idx[0], idx[1], v)), MatrixType.COO)
        if leaves == "1":
            exact = oracle.host_solve(s._factor(), b).astype(ext)
            for _ in range(3):
                r = b - np.add.reduceat(a[:, None] * exact[j], first, axis=0)
                exact = exact + oracle.host_solve(s._factor(), r.astype(np.float64))
        bt = torch.tensor(b, device=DEV)
        xt = torch.zeros_like(bt)
        s.solve(bt, xt)
        torch.cuda.synchronize()
        s._check()
        errors[leaves] = float(np.linalg.norm((xt.cpu().numpy() - exact).astype(np.float64)))
    assert errors["1"] <= 1.04 * errors["0"], errors["1"] / errors["0"]
