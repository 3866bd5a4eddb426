"""The multi-step 2D kernel's tiling fits what the kernel assumes (rows in LDS, width of a
row, halo within the domain) over degenerate, ragged and huge extents."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not present")


def test_tiling(tmp_path):
    exe = str(tmp_path / "tile_rules")
    subprocess.run(["g++", "-std=c++17", "-O2", "-I", os.path.join(ROOT, "include"), "-I",
                    os.path.join(ROOT, "metalbm_amd", "csrc"),
                    os.path.join(ROOT, "tests", "native", "tile_rules.cpp"), "-o", exe],
                   check=True, timeout=300)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout
