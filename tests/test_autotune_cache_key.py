"""A cache line timed with other kernels and plans (a key without their number,
or with another) is not applied."""
import pytest

torch = pytest.importorskip("torch")

from cholespy_amd import CholeskySolverF, MatrixType, workloads

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda")


def test_entries_of_other_plans_are_not_used(tmp_path):
    n, faces = workloads.icosphere(3)
    v, idx = workloads.mesh_laplacian(n, faces, 2.0)

    def solver():
        return CholeskySolverF(n, *(torch.tensor(a, device=DEV) for a in (idx[0], idx[1], v)), MatrixType.COO)

    cache = tmp_path / "tune.txt"
    key = solver().autotune(3, cache=str(cache))["key"]
    line = cache.read_text().strip().splitlines()[-1]
    parts = key.split("-")
    cu = next(i for i, p in enumerate(parts) if p.startswith("cu"))
    assert solver().autotune(3, cache=str(cache))["source"] == "cached"
    for other in ("-".join(parts[:cu + 1]), "-".join(parts[:cu + 1]) + "-p0"):
        cache.write_text(line.replace(key, other) + "\n")
        assert solver().autotune(3, cache=str(cache), write=False)["source"] == "tuned", other
