"""A chain of 2,327 rows as blocks of the two passes (no dense top, which would
take it), with the default and the largest chain caps, against the oracle. The
pattern has the chain; a unit shift keeps kappa ~ 13 (tolerances of the other
parity tests)."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from cholespy_amd import CholeskySolverD, CholeskySolverF, MatrixType, workloads
from oracle import oracle

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda")
TOL = {np.float32: 2e-5, np.float64: 1e-12}


@pytest.mark.parametrize("max_block", [0, 4096])
@pytest.mark.parametrize("cls,dtype", [(CholeskySolverF, np.float32), (CholeskySolverD, np.float64)])
def test_chain_blocks(cls, dtype, max_block, monkeypatch):
    monkeypatch.setenv("CHOLESPY_DENSE_TOP", "0")
    if max_block:
        monkeypatch.setenv("CHOLESPY_MAX_BLOCK", str(max_block))
    n = 40 ** 3
    v, idx = workloads.grid3d_laplacian(40, 1.0)
    s = cls(n, *(torch.tensor(a, device=DEV) for a in (idx[0], idx[1], v)), MatrixType.COO)
    plan = s._plan_arrays()
    assert not (plan["fwd_task"][:, 3] == 4).any()
    assert np.diff(plan["start"]).max() > (2048 if max_block else 1024)
    for k in (3, 9, 32):
        b = np.random.default_rng(k).standard_normal((n, k)).astype(dtype)
        bt = torch.tensor(b, device=DEV)
        xt = torch.zeros_like(bt)
        s.solve(bt, xt)
        torch.cuda.synchronize()
        s._check()
        ref = oracle.solve(s._factor(), b, dtype)
        assert np.abs(xt.cpu().numpy() - ref).max() / np.abs(ref).max() < TOL[dtype], k
