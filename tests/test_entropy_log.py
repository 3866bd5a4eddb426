"""The entropic solve's logarithms, compiled for the host, against the 80-bit library
logarithm: down to the smallest positive number, around 1 and at or below 0."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIP = "/opt/rocm/include"

pytestmark = pytest.mark.skipif(
    shutil.which("g++") is None or not os.path.exists(os.path.join(HIP, "hip", "hip_runtime.h")),
    reason="g++ or the HIP headers not present")


def test_logarithms(tmp_path):
    exe = str(tmp_path / "entropy_log")
    subprocess.run(["g++", "-std=c++17", "-O2", "-ffp-contract=off", "-D__HIP_PLATFORM_AMD__",
                    "-I", HIP, "-I", os.path.join(ROOT, "metalbm_amd", "csrc"),
                    os.path.join(ROOT, "tests", "native", "entropy_log.cpp"), "-o", exe],
                   check=True, timeout=300)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    print(r.stdout)
    assert r.returncode == 0, r.stdout
