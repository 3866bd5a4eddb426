"""The entropic step's single-precision look at a cell (largest |n| / f, smallest f)
decides only what FP64 would decide the same way: cells that are not a number."""
import numpy as np
import pytest

from metalbm_amd import (AlphaMode, Algorithm, CollisionType, Config, ForcingSchemeType,
                         LatticeType, Precision)

pytestmark = pytest.mark.gpu

D2Q9, D3Q27 = LatticeType.D2Q9, LatticeType.D3Q27


def handle(lat, shape, numbers, mode=AlphaMode.NEWTON):
    return Algorithm(Config(
        lattice=lat, collision=CollisionType.ELBM, forcing_scheme=ForcingSchemeType.None_,
        nx=shape[0], ny=shape[1], nz=shape[2], tau=0.6, storage=numbers[0], compute=numbers[1],
        shifted=numbers[2], alpha_mode=mode))


@pytest.mark.parametrize("mode", [AlphaMode.NEWTON, AlphaMode.NEWTON_RESIDUAL,
                                  AlphaMode.WARM_RESIDUAL], ids=lambda m: m.name)
@pytest.mark.parametrize("lat,shape", [(D2Q9, (24, 20, 1)), (D3Q27, (10, 9, 8)),
                                       (D2Q9, (520, 512, 1)), (D3Q27, (41, 40, 42))],
                         ids=["D2Q9", "D3Q27", "D2Q9-large", "D3Q27-large"])
def test_not_a_number_counts_as_fallback(lat, shape, mode):
    """One population that is not a number spoils one cell's moments; its solve fails
    into alpha = 2 and shows in the counters of every solver and size of domain."""
    print("case not a number", lat.name, shape, mode.name, flush=True)
    with handle(lat, shape, (Precision.F32, Precision.F32, True), mode) as a:
        a.init_noise(1.0, 0.0, 1)
        f = a.populations()
        f[3, a.N // 2] = np.nan
        a.set_populations(f)
        a.iterate(1)
        st = a.elbm_stats()
        alpha = a.alpha()
    print(st, flush=True)
    assert (alpha == 2.0).all()
    assert st["fallback"] == 1 and st["small"] == a.N - 1
