"""The dense block values formed on the GPU (block_inverse.hip), at the sizes
where its paths change: blocks inverted in LDS (up to 64 rows) and through
tile products (more), whole and partial 64-row tiles and doublings, and R rows
beyond one 64-row chunk. Solves of both precisions against the oracle on the
same factor; the systems are diagonally dominant (kappa < 10), so the
tolerances are those of the other parity tests."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from cholespy_amd import CholeskySolverD, CholeskySolverF, MatrixType
from oracle import oracle

pytestmark = pytest.mark.gpu

TOL = {np.float32: 2e-5, np.float64: 1e-12}


def _arrow(heads, size, border):
    """`heads` dense diagonal blocks of `size` rows, all coupled to a dense
    border: blocks of `size` columns with `border` R rows each."""
    n = heads * size + border
    rng = np.random.default_rng(size * 1000 + border)
    a = np.zeros((n, n))
    for h in range(heads):
        s = slice(h * size, (h + 1) * size)
        a[s, s] = rng.uniform(-1, 1, (size, size))
        a[heads * size:, s] = rng.uniform(-1, 1, (border, size))
    a[heads * size:, heads * size:] = rng.uniform(-1, 1, (border, border))
    a = np.tril(a, -1)
    a = a + a.T
    np.fill_diagonal(a, 1.2 * np.abs(a).sum(1) + 1.0)
    i, j = np.nonzero(np.tril(a))
    return n, i, j, a[i, j]


@pytest.mark.parametrize("heads,size,border", [(0, 0, 1), (0, 0, 63), (0, 0, 64), (0, 0, 65), (0, 0, 128), (0, 0, 129),
                                               (0, 0, 300), (3, 7, 64), (3, 20, 65), (2, 64, 130), (2, 65, 40),
                                               (2, 100, 200), (1, 257, 191)])
@pytest.mark.parametrize("cls,dtype", [(CholeskySolverF, np.float32), (CholeskySolverD, np.float64)])
def test_block_values_match_oracle(heads, size, border, cls, dtype, monkeypatch):
    monkeypatch.setenv("CHOLESPY_DENSE_TOP", "0")
    n, i, j, v = _arrow(heads, size, border)
    dev = torch.device("cuda")
    s = cls(n, torch.tensor(i, device=dev), torch.tensor(j, device=dev), torch.tensor(v, device=dev), MatrixType.COO)
    rng = np.random.default_rng(n)
    for k in (3, 17):
        b = rng.standard_normal((n, k)).astype(dtype)
        bt = torch.tensor(b, device=dev)
        xt = torch.zeros_like(bt)
        s.solve(bt, xt)
        torch.cuda.synchronize()
        s._check()
        ref = oracle.solve(s._factor(), b, dtype)
        assert np.abs(xt.cpu().numpy() - ref).max() / np.abs(ref).max() < TOL[dtype], k
