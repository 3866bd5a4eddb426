"""The GPU tests that compare the kernels of several steps with those of one run domains for
which the automatic choice takes the former: both widths of 2D tiles, five steps and FP64's
three among them, and the 3D kernel in every 3D case."""
import os
import shutil
import subprocess

import pytest

import march_cases
import test_gpu_call_split as split
import test_gpu_tile as tile
from metalbm_amd import LatticeType

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ROWS = {"F64": (71, 17), "F32": (142, 35), "F16": (284, 71)}  # rows of 16 and 64 cells in LDS

pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not present")


@pytest.fixture(scope="module")
def choice(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("choice") / "step_choice")
    subprocess.run(["g++", "-std=c++17", "-O2", "-I", os.path.join(ROOT, "include"), "-I",
                    os.path.join(ROOT, "metalbm_amd", "csrc"),
                    os.path.join(ROOT, "tests", "native", "step_choice.cpp"), "-o", exe],
                   check=True, timeout=300)

    def run(*args):
        r = subprocess.run([exe, *map(str, args)], capture_output=True, text=True, timeout=60)
        assert r.returncode == 0
        return [int(v) for v in r.stdout.split()]
    return run


def tile_of(choice, shape, storage, equilibrium):
    return tuple(choice("tile", *shape, *ROWS[storage], int(storage == "F64"),
                        int(equilibrium == tile.EXACT)))


def test_2d_cases_take_tiles(choice):
    taken = {}
    for shape, _, _, equilibrium, numbers in tile.CASES:
        taken[shape] = tile_of(choice, shape, numbers[0].name, equilibrium)
    for c in split.CASES:
        if c[0] == LatticeType.D2Q9:
            taken[c[1]] = tile_of(choice, c[1], c[5], c[4])
    for shape, (wide, steps) in taken.items():
        assert steps >= 2, shape
    assert {(0, 5), (1, 5), (1, 3)} <= set(taken.values()), taken


def test_3d_cases_take_two_steps(choice):
    for lattice, shape, scheme, force, equilibrium, _, _, _ in split.CASES:
        if lattice == LatticeType.D2Q9:
            continue
        c = march_cases.case(lattice, shape, scheme, force, equilibrium, True)
        assert choice("march", *shape, *march_cases.kernel_of(c)) == [1], shape
