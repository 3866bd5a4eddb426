"""Single precision with the product equilibrium has no drift of the momentum.

Velocities of decaying noise after some steps, in FP32 and in FP64 arithmetic from the same
populations.  The equilibrium's weights carry one common rounding of 7.5e-9 (1/9 in single
precision), which adds that times omega_eq of the momentum a collision, always one way;
the other roundings should have no preferred sign and grow with the square root of the
steps.  As much again is allowed for them: omega_eq 2^-26 a collision."""
import numpy as np
import pytest

from metalbm_amd import (Algorithm, Config, EquilibriumType, ForceType, ForcingSchemeType,
                         LatticeType, Precision)

pytestmark = pytest.mark.gpu

D2Q9, D3Q27 = LatticeType.D2Q9, LatticeType.D3Q27
STEPS = 24


@pytest.mark.parametrize("tau", [0.6, 0.8])
@pytest.mark.parametrize("lat,n", [(D2Q9, (300, 290, 1)), (D3Q27, (70, 66, 60))],
                         ids=["D2Q9", "D3Q27"])
def test_product_equilibrium(lat, n, tau):
    print("case momentum", lat.name, tau, flush=True)

    def run(precision, shifted, f0=None):
        with Algorithm(Config(lattice=lat, nx=n[0], ny=n[1], nz=n[2], tau=tau,
                              forcing_scheme=ForcingSchemeType.None_, force=ForceType.None_,
                              equilibrium=EquilibriumType.Exact, storage=precision,
                              compute=precision, shifted=shifted)) as a:
            if f0 is None:
                a.init_noise(1.0, 1e-2, 5)
                return a.populations()
            a.set_populations(f0)
            a.iterate(STEPS, store=True)
            return a.store_fields()[1]
    f0 = run(Precision.F32, True)
    got, want = run(Precision.F32, True, f0), run(Precision.F64, False, f0)
    off = np.linalg.norm(got - want) / np.linalg.norm(want)
    print(f"velocities off by {off:.2e}", flush=True)
    assert off <= STEPS * 2.0 ** -26 / tau
