"""Memory for the list of an entropic step's cells (4 bytes a cell) is taken by the alpha
modes that list cells, and only by those."""
import ctypes
import os

import numpy as np
import pytest

from metalbm_amd import (AlphaMode, Algorithm, CollisionType, Config, ForcingSchemeType,
                         LatticeType, Precision)

pytestmark = pytest.mark.gpu

D2Q9, D3Q19 = LatticeType.D2Q9, LatticeType.D3Q19
F64, F32 = (Precision.F64, Precision.F64, False), (Precision.F32, Precision.F32, True)
LIST_FREE = [(D2Q9, (4096, 4096, 1), F64, AlphaMode.NEWTON),
             (D2Q9, (4096, 4096, 1), F32, AlphaMode.NEWTON_RESIDUAL),
             (D3Q19, (256, 256, 256), F64, AlphaMode.NEWTON)]


def config(lat, n, numbers, mode):
    return Config(lattice=lat, collision=CollisionType.ELBM,
                  forcing_scheme=ForcingSchemeType.None_, nx=n[0], ny=n[1], nz=n[2], tau=0.5005,
                  storage=numbers[0], compute=numbers[1], shifted=numbers[2], alpha_mode=mode)


def free_memory():
    for lib in ("/opt/rocm/lib/libamdhip64.so", "libamdhip64.so"):
        if os.path.sep not in lib or os.path.exists(lib):
            H = ctypes.CDLL(lib)
            break
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert H.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


@pytest.mark.parametrize("lat,n,numbers,mode", LIST_FREE,
                         ids=[f"{c[0].name}-{c[2][0].name}-{c[3].name}" for c in LIST_FREE])
def test_no_list_where_none_is_read(lat, n, numbers, mode):
    print("case list memory", lat.name, numbers[0].name, mode.name, flush=True)
    with Algorithm(config(D2Q9, (16, 16, 1), F64, AlphaMode.NEWTON)):
        before = free_memory()  # the runtime's own memory is in use by now
        with Algorithm(config(lat, n, numbers, mode)) as a:
            taken = before - free_memory()
            size = 8 if numbers is F64 else 4
            state = (2 * a.Q + 1) * a.N * size  # both lattices and the alpha field
            print(f"{taken / 2 ** 20:.1f} MiB taken, {state / 2 ** 20:.1f} of state", flush=True)
            assert taken - state < 2 * a.N


def test_list_of_a_mode_set_later():
    """A mode that lists cells, set after creation, solves as in a handle created with it."""
    print("case list of a mode set later", flush=True)
    out = []
    for mode in (AlphaMode.NEWTON, AlphaMode.NEWTON_RESIDUAL):
        with Algorithm(config(D2Q9, (520, 512, 1), F32, mode)) as a:
            a.init_noise(1.0, 6e-2, 5)
            a.set_alpha_mode(AlphaMode.NEWTON)
            a.iterate(3)
            out.append((a.populations(), a.alpha(), a.elbm_stats()))
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])
    assert out[0][2] == out[1][2]
