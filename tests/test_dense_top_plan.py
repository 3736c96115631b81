"""CPU check of plans with a dense top: the choice of its rows, the numbering,
the task lists, the panels of the two products and the tile products that form
the inverse, by emulation (tests/dense_top_emulator.cpp, built here with g++).
Connected systems, forests of several trees and a postorder's random
renumbering, with caps from one row to the whole system."""
import shutil
import subprocess
from pathlib import Path

import numpy as np
import pytest

from cholespy_amd import CholeskySolverD, MatrixType, workloads

ROOT = Path(__file__).resolve().parents[1]
DEVICE = ROOT / "cholespy_amd" / "csrc" / "device"


@pytest.fixture(scope="module")
def emulator(tmp_path_factory):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("g++ is not available")
    exe = tmp_path_factory.mktemp("top") / "dense_top_emulator"
    subprocess.run([cxx, "-O2", "-std=c++17", "-pthread", "-I", str(DEVICE),
                    str(ROOT / "tests" / "dense_top_emulator.cpp"), str(DEVICE / "block_plan.cpp"),
                    str(DEVICE / "dense_top_plan.cpp"), "-o", str(exe)], check=True)
    return exe


def _forest(*grids):
    """Unconnected grids, as one system."""
    n, values, rows, cols = 0, [], [], []
    for nx, ny in grids:
        v, idx = workloads.grid2d_laplacian(nx, ny, 0.5)
        values.append(v)
        rows.append(idx[0] + n)
        cols.append(idx[1] + n)
        n += nx * ny
    return n, np.concatenate(values), np.stack([np.concatenate(rows), np.concatenate(cols)])


def _mesh(level):
    n, f = workloads.icosphere(level)
    return (n,) + workloads.mesh_laplacian(n, f, 2.0)


CASES = {
    "one": lambda: _forest((1, 1)),
    "grid5x13": lambda: _forest((5, 13)),
    "grid61x47": lambda: _forest((61, 47)),
    "ico4": lambda: _mesh(4),
    "cube13": lambda: (13 ** 3,) + workloads.grid3d_laplacian(13, 0.5),
    "forest": lambda: _forest((30, 31), (3, 3), (40, 17), (1, 1), (16, 16), (25, 25)),
    "dust": lambda: _forest((20, 20), *[(1, 1)] * 70),
}


@pytest.fixture(scope="module")
def factors(tmp_path_factory):
    out, d = {}, tmp_path_factory.mktemp("top_factors")
    for name, make in CASES.items():
        n, values, idx = make()
        fac = CholeskySolverD(n, idx[0], idx[1], values, MatrixType.COO)._factor()
        out[name] = d / f"{name}.bin"
        with open(out[name], "wb") as fh:
            fh.write(np.array([n, len(fac["rowidx"])], dtype=np.int64).tobytes())
            for key, dt in (("colptr", np.int32), ("rowidx", np.int32), ("val", np.float64)):
                fh.write(np.ascontiguousarray(fac[key], dtype=dt).tobytes())
    return out


@pytest.mark.parametrize("shuffle", [0, 1])
@pytest.mark.parametrize("rows", [0, 1, 15, 64, 200, 900, 7168])
@pytest.mark.parametrize("case", sorted(CASES))
def test_top_schedule_and_inverse(case, rows, shuffle, factors, emulator):
    for kind, mib in (("narrow", 4096), ("wide", 4)):
        res = subprocess.run([str(emulator), str(factors[case]), kind, str(rows), str(shuffle), str(mib)], capture_output=True,
                             text=True, timeout=120)
        assert res.returncode == 0, (case, kind, rows, shuffle, res.stdout + res.stderr)
        print(kind, res.stdout.strip())


def test_inverse_is_stored_where_it_is_nonzero(factors, emulator):
    """A 61 x 47 grid as one top: a dense square would take 180 x 180 units."""
    res = subprocess.run([str(emulator), str(factors["grid61x47"]), "narrow", "7168", "0", "4096"], capture_output=True, text=True)
    assert "top 2867" in res.stdout and " units 2122 tiles 264 " in res.stdout, res.stdout


def test_forest_top_has_a_block_per_tree(factors, emulator):
    res = subprocess.run([str(emulator), str(factors["forest"]), "narrow", "7168", "0", "4096"], capture_output=True, text=True)
    assert "in 6 blocks of 6, trees 6" in res.stdout, res.stdout
    # Too many trees for a top of all rows: fewer levels, or none.
    res = subprocess.run([str(emulator), str(factors["dust"]), "narrow", "7168", "0", "4096"], capture_output=True, text=True)
    assert "ok" in res.stdout and "top 470" not in res.stdout, res.stdout


def test_groups_of_bounded_work(factors, emulator):
    """32 KiB a tile, twice: the forest's six trees in several groups, each within 8 MiB."""
    res = subprocess.run([str(emulator), str(factors["forest"]), "narrow", "7168", "0", "8"], capture_output=True, text=True)
    assert res.returncode == 0 and " groups 2 " in res.stdout or " groups 3 " in res.stdout, res.stdout
