"""The two-step kernel's tiling fits what the kernel assumes (LDS, registers,
packed indexes, grid) over degenerate, ragged and huge extents, and the automatic
choice takes it for the shapes that tests/test_gpu_march.py runs."""
import os
import shutil
import subprocess

import pytest

from march_cases import CASES, kernel_of

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not present")


def test_tiling(tmp_path):
    exe = str(tmp_path / "march_rules")
    subprocess.run(["g++", "-std=c++17", "-O2", "-I", os.path.join(ROOT, "include"), "-I",
                    os.path.join(ROOT, "metalbm_amd", "csrc"),
                    os.path.join(ROOT, "tests", "native", "march_rules.cpp"), "-o", exe],
                   check=True, timeout=300)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout
    for c in CASES:
        r = subprocess.run([exe, *map(str, c["shape"] + kernel_of(c))], capture_output=True,
                           text=True, timeout=60)
        assert r.stdout.strip() == "1", c
