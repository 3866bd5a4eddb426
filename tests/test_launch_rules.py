"""The split of a call's steps over launches of the multi-step 2D kernel: each takes between
one step and what its tiling allows, their sum is the call, and their number has its parity,
up to the largest call (signed overflow is an error of the build)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not present")


def test_launches(tmp_path):
    exe = str(tmp_path / "launch_rules")
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Werror=sequence-point", "-fsanitize=signed-integer-overflow",
                    "-fno-sanitize-recover=all",
                    "-I", os.path.join(ROOT, "include"), "-I",
                    os.path.join(ROOT, "metalbm_amd", "csrc"),
                    os.path.join(ROOT, "tests", "native", "launch_rules.cpp"), "-o", exe],
                   check=True, timeout=300)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout
