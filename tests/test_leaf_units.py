"""Leaf tasks run by single wavefronts at wide right-hand sides (trsv_panel.hip):
inside the panel launches, and in launches of their own where a batch has many.
The widths sit at the ends of the 16- and 32-column tiles; the oracle solves
with the same factor (kappa < 10, the tolerances of the other parity tests)."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from cholespy_amd import BatchedSolverD, BatchedSolverF, CholeskySolverD, CholeskySolverF, MatrixType, workloads
from oracle import oracle

pytestmark = pytest.mark.gpu

TOL = {np.float32: 2e-5, np.float64: 1e-12}


@pytest.mark.parametrize("system", ["grid2", "grid3", "mesh"])
@pytest.mark.parametrize("cls,dtype", [(CholeskySolverF, np.float32), (CholeskySolverD, np.float64)])
def test_fused_units(system, cls, dtype, monkeypatch):
    monkeypatch.setenv("CHOLESPY_DENSE_TOP", "0")
    if system == "grid2":
        n, (v, idx) = 97 * 61, workloads.grid2d_laplacian(97, 61, 1.0)
    elif system == "grid3":
        n, (v, idx) = 17 ** 3, workloads.grid3d_laplacian(17, 1.0)
    else:
        n, faces = workloads.icosphere(4)
        v, idx = workloads.mesh_laplacian(n, faces, 1.0)
    dev = torch.device("cuda")
    s = cls(n, torch.tensor(idx[0], device=dev), torch.tensor(idx[1], device=dev), torch.tensor(v, device=dev),
            MatrixType.COO)
    rng = np.random.default_rng(n)
    for k in (16, 17, 31, 32, 33, 64, 65, 127, 128):
        b = rng.standard_normal((n, k)).astype(dtype)
        bt = torch.tensor(b, device=dev)
        xt = torch.zeros_like(bt)
        for _ in range(2):   # the second solve starts from what the first one left
            s.solve(bt, xt)
        torch.cuda.synchronize()
        s._check()
        ref = oracle.solve(s._factor(), b, dtype)
        assert np.abs(xt.cpu().numpy() - ref).max() / np.abs(ref).max() < TOL[dtype], k


@pytest.mark.parametrize("cls,dtype", [(BatchedSolverF, np.float32), (BatchedSolverD, np.float64)])
def test_units_in_their_own_launch(cls, dtype):
    """A batch with more than 16,384 leaf units."""
    sizes = [(45 + i % 3, 44 + i % 5) for i in range(80)]
    systems = [workloads.grid2d_laplacian(nx, ny, 1.0) for nx, ny in sizes]
    batch = cls([(nx * ny, i[0], i[1], v, MatrixType.COO) for (nx, ny), (v, i) in zip(sizes, systems)])
    tasks = batch._plan_arrays()
    level = tasks["level_fwd"][tasks["fwd_task_wide"][:, 0]]
    assert (level == 0).sum() * 4 > 16384
    ks = [(0, 1, 16, 17, 33, 128)[i % 6] for i in range(len(sizes))]
    rng = np.random.default_rng(1)
    bs = [rng.standard_normal((nx * ny, k)).astype(dtype) for (nx, ny), k in zip(sizes, ks)]
    b = torch.tensor(np.concatenate([x.ravel() for x in bs]), device="cuda")
    x = torch.zeros_like(b)
    for _ in range(2):
        batch.solve(ks, b, x)
    torch.cuda.synchronize()
    batch._check()
    got, at = x.cpu().numpy(), 0
    for i, ((nx, ny), k) in enumerate(zip(sizes, ks)):
        n = nx * ny
        if k and i % 5 == 0:
            ref = oracle.solve(batch._factor(i), bs[i], dtype)
            assert np.abs(got[at:at + n * k].reshape(n, k) - ref).max() / np.abs(ref).max() < TOL[dtype], (i, k)
        at += n * k
