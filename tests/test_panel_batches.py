"""The backward pass of the panel kernels (more than four right-hand sides):
batches of reduction steps that end before, at and after the last step, tiles
that end inside a row, diagonal pieces, and row indices too many for LDS.
The systems are diagonally dominant (kappa < 10); the oracle solves with the
same factor, and the tolerances are those of the other parity tests."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from cholespy_amd import CholeskySolverD, CholeskySolverF, MatrixType, workloads
from oracle import oracle

pytestmark = pytest.mark.gpu

TOL = {np.float32: 2e-5, np.float64: 1e-12}
DEV = torch.device("cuda")


def _check(s, n, k, dtype):
    b = np.random.default_rng(n + k).standard_normal((n, k)).astype(dtype)
    bt = torch.tensor(b, device=DEV)
    xt = torch.zeros_like(bt)
    s.solve(bt, xt)
    torch.cuda.synchronize()
    s._check()
    ref = oracle.solve(s._factor(), b, dtype)
    assert np.abs(xt.cpu().numpy() - ref).max() / np.abs(ref).max() < TOL[dtype], (n, k)


@pytest.mark.parametrize("max_block", [3, 16, 50, 64, 200])
@pytest.mark.parametrize("cls,dtype", [(CholeskySolverF, np.float32), (CholeskySolverD, np.float64)])
def test_batches_of_every_length(max_block, cls, dtype, monkeypatch):
    monkeypatch.setenv("CHOLESPY_DENSE_TOP", "0")
    monkeypatch.setenv("CHOLESPY_MAX_BLOCK", str(max_block))
    v, idx = workloads.grid3d_laplacian(11, 1.0)
    n = 11 ** 3
    s = cls(n, *(torch.tensor(a, device=DEV) for a in (idx[0], idx[1], v)), MatrixType.COO)
    for k in (5, 16, 17, 32, 33, 50, 64, 65, 97, 128):
        _check(s, n, k, dtype)


def test_more_rows_than_lds_indices(monkeypatch):
    """A dense system cut into blocks of at most 64 rows: the first has 4,136 below."""
    monkeypatch.setenv("CHOLESPY_DENSE_TOP", "0")
    monkeypatch.setenv("CHOLESPY_MAX_BLOCK", "40")
    monkeypatch.setenv("CHOLESPY_SPLIT_ENTRIES", "0")
    n = 4200
    c = np.random.default_rng(3).uniform(-1, 1, n)
    a = np.outer(c, c) / n
    a[np.arange(n), np.arange(n)] += 1.0
    rows, cols = np.indices((n, n)).reshape(2, -1)
    s = CholeskySolverF(n, *(torch.tensor(x, device=DEV) for x in (rows, cols, a.ravel())), MatrixType.COO)
    arrays = s._plan_arrays()
    assert np.diff(arrays["rptr"]).max() > 4096
    for k in (7, 40):
        _check(s, n, k, np.float32)
