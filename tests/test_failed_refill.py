"""A refill of a handle's values that fails part way (its work memory cannot be
had: the bound CHOLESPY_FILL_MIB, set to nothing on the host, stands in for
that) leaves no handle that solves with what is there: solves raise until a
refactorisation succeeds, and are right again after it."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from cholespy_amd import CholeskySolverD, CholeskySolverF, MatrixType, workloads
from oracle import oracle

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda")
TOL = {np.float32: 2e-5, np.float64: 1e-12}


def _right(s, n, dtype):
    b = np.random.default_rng(n).standard_normal((n, 3)).astype(dtype)
    bt = torch.tensor(b, device=DEV)
    xt = torch.zeros_like(bt)
    s.solve(bt, xt)
    torch.cuda.synchronize()
    s._check()
    ref = oracle.solve(s._factor(), b, dtype)
    assert np.abs(xt.cpu().numpy() - ref).max() / np.abs(ref).max() < TOL[dtype]


def _refuses(s, n, dtype):
    bt = torch.zeros((n, 3), device=DEV, dtype=torch.float32 if dtype == np.float32 else torch.float64)
    with pytest.raises(RuntimeError, match="before the factor was uploaded"):
        s.solve(bt, torch.zeros_like(bt))
    if dtype == np.float32:
        with pytest.raises(RuntimeError, match="before the factor was uploaded"):
            s._solve_refined(bt.double(), torch.zeros_like(bt.double()), 1)


@pytest.mark.parametrize("cls,dtype", [(CholeskySolverF, np.float32), (CholeskySolverD, np.float64)])
@pytest.mark.parametrize("m", [9, 24])   # a whole top; levels, large blocks and a top
def test_failed_refactorize(m, cls, dtype, monkeypatch):
    n = m ** 3
    v, idx = workloads.grid3d_laplacian(m, 1.0)
    s = cls(n, *(torch.tensor(a, device=DEV) for a in (idx[0], idx[1], v)), MatrixType.COO)
    _right(s, n, dtype)
    new = v.copy()
    new[:n] += 0.5
    monkeypatch.setenv("CHOLESPY_FILL_MIB", "0")
    with pytest.raises(RuntimeError, match="out of memory"):
        s.refactorize(torch.tensor(new, device=DEV))
    _refuses(s, n, dtype)
    monkeypatch.delenv("CHOLESPY_FILL_MIB")
    s.refactorize(torch.tensor(new, device=DEV))
    _right(s, n, dtype)


def test_failed_constructor(monkeypatch):
    monkeypatch.setenv("CHOLESPY_FILL_MIB", "0")
    v, idx = workloads.grid3d_laplacian(9, 1.0)
    with pytest.raises(RuntimeError, match="out of memory"):
        CholeskySolverF(729, *(torch.tensor(a, device=DEV) for a in (idx[0], idx[1], v)), MatrixType.COO)


def test_failed_autotune(monkeypatch, tmp_path):
    """A candidate plan whose values cannot be formed."""
    n = 24 ** 3
    v, idx = workloads.grid3d_laplacian(24, 1.0)
    s = CholeskySolverF(n, *(torch.tensor(a, device=DEV) for a in (idx[0], idx[1], v)), MatrixType.COO)
    monkeypatch.setenv("CHOLESPY_FILL_MIB", "0")
    with pytest.raises(RuntimeError, match="out of memory"):
        s.autotune(3, cache=str(tmp_path / "cache.txt"))
    _refuses(s, n, np.float32)
    monkeypatch.delenv("CHOLESPY_FILL_MIB")
    s.refactorize(torch.tensor(v, device=DEV))
    _right(s, n, np.float32)


@pytest.mark.parametrize("cls,dtype", [(CholeskySolverF, np.float32), (CholeskySolverD, np.float64)])
def test_refill_in_groups(cls, dtype, monkeypatch):
    """Less work memory than all blocks together take: one group after another
    (the tops of three unconnected parts, and the large blocks below them)."""
    monkeypatch.setenv("CHOLESPY_FILL_MIB", "48")
    n, values, rows, cols = 0, [], [], []
    for m in (9, 21, 24):
        v, idx = workloads.grid3d_laplacian(m, 1.0)
        values.append(v)
        rows.append(idx[0] + n)
        cols.append(idx[1] + n)
        n += m ** 3
    s = cls(n, *(torch.tensor(np.concatenate(a), device=DEV) for a in (rows, cols, values)), MatrixType.COO)
    assert (s._plan_arrays()["fwd_task"][:, 3] == 4).any()
    _right(s, n, dtype)
    s.refactorize(torch.tensor(np.concatenate(values), device=DEV))
    _right(s, n, dtype)
