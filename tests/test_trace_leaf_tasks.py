"""The task timeline holds every task of both passes, leaf tasks run by single
wavefronts (more than 16 right-hand sides) among them: in the block launches
and, for a batch of many, in launches of their own."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from cholespy_amd import BatchedSolverF, CholeskySolverD, CholeskySolverF, MatrixType, workloads

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda")


def _check(s, run):
    s._set_trace(True)
    run()
    torch.cuda.synchronize()
    plan = s._plan_arrays()
    for forward in (True, False):
        tasks = plan[("fwd" if forward else "bwd") + "_task_wide"]
        t = np.asarray(s._trace(forward)).reshape(-1, 4)[:len(tasks)].astype(np.int64)
        assert (t[:, 0] > 0).all() and (t[:, 2] >= t[:, 0]).all(), forward
        assert t[:, 2].max() - t[:, 0].min() < 10 ** 8, "a second in 10 ns ticks"
    s._set_trace(False)


@pytest.mark.parametrize("top", ["0", "2000"])
@pytest.mark.parametrize("cls,dtype", [(CholeskySolverF, torch.float32), (CholeskySolverD, torch.float64)])
def test_single_system(top, cls, dtype, monkeypatch):
    monkeypatch.setenv("CHOLESPY_DENSE_TOP", top)
    n = 151 * 97
    v, idx = workloads.grid2d_laplacian(151, 97, 1.0)
    s = cls(n, *(torch.tensor(a, device=DEV) for a in (idx[0], idx[1], v)), MatrixType.COO)
    for k in (8, 20, 100):
        b = torch.ones(n, k, device=DEV, dtype=dtype)
        _check(s, lambda: s.solve(b, torch.zeros_like(b)))


def test_batch_with_leaf_launches():
    sizes = [(45 + i % 3, 44 + i % 5) for i in range(80)]
    systems = [workloads.grid2d_laplacian(nx, ny, 1.0) for nx, ny in sizes]
    batch = BatchedSolverF([(nx * ny, i[0], i[1], v, MatrixType.COO) for (nx, ny), (v, i) in zip(sizes, systems)])
    ks = [1 + 127 * (i % 2) for i in range(80)]
    b = torch.ones(sum(nx * ny * k for (nx, ny), k in zip(sizes, ks)), device=DEV)
    _check(batch, lambda: batch.solve(ks, b, torch.zeros_like(b)))
