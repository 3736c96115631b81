"""Refined solves (x += correction) at widths that do not fill the dense
product's tiles: every entry of x takes each correction exactly once. A whole
small system and one with a top between the passes, against the FP64 host
solve on the same factor.

Tolerances: the systems have kappa <= 9, and an FP32 solve is within 2e-5 (the
other parity tests' bound), so one correction leaves at most 4e-10 and two at
most 8e-15, where the FP64 residual's rounding (about kappa * 1e-16) takes
over: 1e-12."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from cholespy_amd import CholeskySolverF, MatrixType, workloads
from oracle import oracle

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda")


@pytest.mark.parametrize("nx,ny", [(20, 21), (151, 97)])
def test_each_correction_is_added_once(nx, ny):
    n = nx * ny
    v, idx = workloads.grid2d_laplacian(nx, ny, 1.0)
    s = CholeskySolverF(n, *(torch.tensor(a, device=DEV) for a in (idx[0], idx[1], v)), MatrixType.COO)
    assert (s._plan_arrays()["fwd_task"][:, 3] == 4).any()
    for k in (5, 16, 17, 31, 32, 33, 49, 50, 63, 65, 80, 81, 97, 127, 128):
        b = np.random.default_rng(k).standard_normal((n, k))
        ref = oracle.host_solve(s._factor(), b)
        bt = torch.tensor(b, device=DEV)
        for steps, tol in ((1, 4e-10), (2, 1e-12)):
            xt = torch.zeros_like(bt)
            s._solve_refined(bt, xt, steps)
            torch.cuda.synchronize()
            s._check()
            err = np.linalg.norm(xt.cpu().numpy() - ref, axis=0) / np.linalg.norm(ref, axis=0)
            assert err.max() < tol, (k, steps, np.nonzero(err >= tol)[0])
        steps, res = s._solve_refined_tol(bt, torch.zeros_like(bt), 1e-12, 6)
        assert res <= 1e-12 and steps <= 3, (k, steps, res)
