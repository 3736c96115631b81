"""Dense top blocks (dense_top.hip): whole systems solved by one product and
tops between the passes, at the sizes where the panels, chunks and tiles end,
for every right-hand-side width class, both precisions, in place, and through
the single passes. The oracle solves with the same factor; the systems are
diagonally dominant (kappa < 10), so the tolerances are those of the other
parity tests."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from cholespy_amd import BatchedSolverD, CholeskySolverD, CholeskySolverF, MatrixType, workloads
from oracle import oracle

pytestmark = pytest.mark.gpu

TOL = {np.float32: 2e-5, np.float64: 1e-12}
DEV = torch.device("cuda")


def _check(s, n, k, dtype, tol, in_place=False):
    b = np.random.default_rng(n + k).standard_normal((n, k) if k else n).astype(dtype)
    bt = torch.tensor(b, device=DEV)
    xt = bt if in_place else torch.zeros_like(bt)
    s.solve(bt, xt)
    torch.cuda.synchronize()
    s._check()
    ref = oracle.solve(s._factor(), b.reshape(n, -1), dtype).reshape(b.shape)
    assert np.abs(xt.cpu().numpy() - ref).max() / np.abs(ref).max() < tol, (n, k)


def _solver(cls, nx, ny):
    v, idx = workloads.grid2d_laplacian(nx, ny, 1.0)
    return nx * ny, cls(nx * ny, *(torch.tensor(a, device=DEV) for a in (idx[0], idx[1], v)), MatrixType.COO)


@pytest.mark.parametrize("nx,ny", [(1, 1), (3, 5), (4, 4), (1, 17), (24, 32), (25, 31), (48, 32), (49, 33)])
@pytest.mark.parametrize("cls,dtype", [(CholeskySolverF, np.float32), (CholeskySolverD, np.float64)])
def test_whole_system(nx, ny, cls, dtype):
    n, s = _solver(cls, nx, ny)
    assert s._plan_info()["fwd_tasks"] == -(-n // 64) and s._plan_info()["bwd_tasks"] == 0
    for k in (0, 1, 3, 4, 5, 16, 17, 33, 64, 65, 128):
        _check(s, n, k, dtype, TOL[dtype])
    _check(s, n, 3, dtype, TOL[dtype], in_place=True)
    _check(s, n, 40, dtype, TOL[dtype], in_place=True)


@pytest.mark.parametrize("rows", [300, 1000, 6400])
@pytest.mark.parametrize("cls,dtype", [(CholeskySolverF, np.float32), (CholeskySolverD, np.float64)])
def test_top_between_the_passes(rows, cls, dtype, monkeypatch):
    monkeypatch.setenv("CHOLESPY_DENSE_TOP", str(rows))
    n, s = _solver(cls, 151, 97)
    tasks = s._plan_arrays()["fwd_task"]
    assert (tasks[:, 3] == 4).any() and s._plan_info()["bwd_tasks"] > 0
    for k in (1, 3, 4, 5, 17, 100):
        _check(s, n, k, dtype, TOL[dtype])
    _check(s, n, 3, dtype, TOL[dtype], in_place=True)
    b = torch.randn(n, 3, device=DEV, dtype=torch.float32 if dtype == np.float32 else torch.float64)
    x, y = torch.zeros_like(b), torch.zeros_like(b)
    s.solve(b, x)
    s._solve_pass(0, b, y)
    s._solve_pass(1, b, y)
    torch.cuda.synchronize()
    assert torch.equal(x, y)


def test_batch_mixes_whole_systems_and_tops():
    """Sixteen systems from 12 to 4,900 rows, some a single product, some with
    a top, with right-hand-side counts of 0 to 70."""
    sizes = [(3, 4), (10, 10), (20, 21), (30, 33), (40, 40), (70, 70), (25, 80), (64, 48)] * 2
    systems = [workloads.grid2d_laplacian(nx, ny, 1.0) for nx, ny in sizes]
    batch = BatchedSolverD([(nx * ny, i[0], i[1], v, MatrixType.COO) for (nx, ny), (v, i) in zip(sizes, systems)])
    rng = np.random.default_rng(4)
    for ks in ([3] * 16, [(7 * i) % 71 for i in range(16)], [i % 5 for i in range(16)]):
        bs = [rng.standard_normal((nx * ny, k)) for (nx, ny), k in zip(sizes, ks)]
        b = torch.tensor(np.concatenate([x.ravel() for x in bs]), device=DEV)
        x = torch.zeros_like(b)
        batch.solve(ks, b, x)
        torch.cuda.synchronize()
        batch._check()
        got, at = x.cpu().numpy(), 0
        for i, ((nx, ny), k) in enumerate(zip(sizes, ks)):
            n = nx * ny
            if k:
                ref = oracle.solve(batch._factor(i), bs[i], np.float64)
                assert np.abs(got[at:at + n * k].reshape(n, k) - ref).max() / np.abs(ref).max() < 1e-12, (i, k)
            at += n * k


@pytest.mark.parametrize("ks", [[5, 17, 18, 19, 31, 6, 32, 16], [4, 33, 34, 47, 66, 7, 125, 64]])
def test_batch_right_hand_sides_of_unequal_tiles(ks):
    """The widest system of a batch sets the tiles of all (2 or 4 of 16
    right-hand sides): rows that end before, inside and at the end of a tile."""
    n = 20 * 21
    v, idx = workloads.grid2d_laplacian(20, 21, 1.0)
    batch = BatchedSolverD([(n, idx[0], idx[1], v, MatrixType.COO)] * len(ks))
    bs = [np.random.default_rng(k).standard_normal((n, k)) for k in ks]
    b = torch.tensor(np.concatenate([x.ravel() for x in bs]), device=DEV)
    x = torch.zeros_like(b)
    batch.solve(ks, b, x)
    torch.cuda.synchronize()
    batch._check()
    got = np.split(x.cpu().numpy(), np.cumsum([n * k for k in ks])[:-1])
    for i, k in enumerate(ks):
        ref = oracle.solve(batch._factor(i), bs[i], np.float64)
        assert np.abs(got[i].reshape(n, k) - ref).max() / np.abs(ref).max() < 1e-12, (i, k)
