"""Panels of the dense top's products that several workgroups share: tops of
more than 96 units of 16 rows, at the widths of each kernel and of its rests,
repeated (the arrival counters start from zero each time), in a graph's replays
and in a batch whose systems differ in their right-hand sides. The oracle
solves with the same factor (kappa < 20; tolerances of the other parity tests)."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from cholespy_amd import BatchedSolverD, BatchedSolverF, CholeskySolverD, CholeskySolverF, MatrixType, workloads
from oracle import oracle

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda")
TOL = {np.float32: 2e-5, np.float64: 1e-12}


@pytest.mark.parametrize("cls,dtype", [(CholeskySolverF, np.float32), (CholeskySolverD, np.float64)])
@pytest.mark.parametrize("nx,ny", [(70, 45), (151, 130)])
def test_segments(nx, ny, cls, dtype):
    n = nx * ny
    v, idx = workloads.grid2d_laplacian(nx, ny, 0.5)
    s = cls(n, *(torch.tensor(a, device=DEV) for a in (idx[0], idx[1], v)), MatrixType.COO)
    plan = s._plan_arrays()
    tops = np.unique(plan["fwd_task"][plan["fwd_task"][:, 3] == 4, 0])
    assert np.diff(plan["start"])[tops].max() > 96 * 16
    for k in (0, 1, 4, 5, 16, 17, 40, 65, 128):
        b = np.random.default_rng(k).standard_normal((n, k) if k else n).astype(dtype)
        bt = torch.tensor(b, device=DEV)
        xs = []
        for _ in range(3):
            xs.append(torch.zeros_like(bt))
            s.solve(bt, xs[-1])
        torch.cuda.synchronize()
        s._check()
        ref = oracle.solve(s._factor(), b.reshape(n, -1), dtype).reshape(b.shape)
        assert np.abs(xs[0].cpu().numpy() - ref).max() / np.abs(ref).max() < TOL[dtype], k
        assert torch.equal(xs[0], xs[1]) and torch.equal(xs[0], xs[2]), k


@pytest.mark.parametrize("cls", [CholeskySolverF, CholeskySolverD])
def test_segments_in_a_graph(cls):
    n = 70 * 45
    v, idx = workloads.grid2d_laplacian(70, 45, 0.5)
    s = cls(n, *(torch.tensor(a, device=DEV) for a in (idx[0], idx[1], v)), MatrixType.COO)
    dtype = torch.float32 if cls is CholeskySolverF else torch.float64
    b = torch.zeros(n, 3, device=DEV, dtype=dtype)
    x, y = torch.zeros_like(b), torch.zeros_like(b)
    s.solve(b, x)
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        s.solve(b, x, stream=stream.cuda_stream)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        s.solve(b, x, stream=stream.cuda_stream)
    for seed in range(4):
        b.copy_(torch.randn(n, 3, generator=torch.Generator().manual_seed(seed)).to(dtype))
        s.solve(b, y)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(x, y), seed


@pytest.mark.parametrize("cls,dtype", [(BatchedSolverF, np.float32), (BatchedSolverD, np.float64)])
def test_segments_in_a_batch(cls, dtype):
    """Fewer than eight systems: tops of any size."""
    sizes = [(70, 45), (12, 10), (61, 53), (90, 80)]
    systems = [workloads.grid2d_laplacian(nx, ny, 0.5) for nx, ny in sizes]
    batch = cls([(nx * ny, i[0], i[1], v, MatrixType.COO) for (nx, ny), (v, i) in zip(sizes, systems)])
    for ks in ([3, 1, 0, 4], [17, 3, 128, 33], [5, 16, 50, 0]):
        bs = [np.random.default_rng(k).standard_normal((nx * ny, k)).astype(dtype) for (nx, ny), k in zip(sizes, ks)]
        b = torch.tensor(np.concatenate([q.ravel() for q in bs]), device=DEV)
        x, y = torch.zeros_like(b), torch.zeros_like(b)
        batch.solve(ks, b, x)
        batch.solve(ks, b, y)
        torch.cuda.synchronize()
        batch._check()
        assert torch.equal(x, y)
        got, at = x.cpu().numpy(), 0
        for i, ((nx, ny), k) in enumerate(zip(sizes, ks)):
            if k:
                ref = oracle.solve(batch._factor(i), bs[i], dtype)
                part = got[at:at + nx * ny * k].reshape(-1, k)
                assert np.abs(part - ref).max() / np.abs(ref).max() < TOL[dtype], (i, k)
            at += nx * ny * k
