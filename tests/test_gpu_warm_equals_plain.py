"""The certified correction from the stored alpha accepts iterates of plain Newton's own, so
with plain Newton as its fallback it ends with the same alpha: in FP32 arithmetic both
modes give the same populations, stored alphas, roots and fallbacks, step after step."""
import numpy as np
import pytest

from metalbm_amd import (AlphaMode, Algorithm, CollisionType, Config, ForceType,
                         ForcingSchemeType, LatticeType, Precision)

pytestmark = pytest.mark.gpu

D2Q9, D3Q19, D3Q27 = LatticeType.D2Q9, LatticeType.D3Q19, LatticeType.D3Q27
CASES = [(D2Q9, (200, 120, 1), 2e-2), (D3Q19, (33, 30, 34), 2e-2), (D3Q27, (21, 20, 18), 5e-2),
         (D3Q27, (41, 40, 42), 2e-2), (D3Q27, (64, 64, 64), 5e-2)]


@pytest.mark.parametrize("lat,n,amp", CASES, ids=[f"{c[0].name}-{c[1][0]}" for c in CASES])
def test_same_results(lat, n, amp):
    print("case warm equals plain", lat.name, n, flush=True)
    out = []
    for mode in (AlphaMode.NEWTON_RESIDUAL, AlphaMode.WARM_RESIDUAL):
        with Algorithm(Config(lattice=lat, collision=CollisionType.ELBM,
                              forcing_scheme=ForcingSchemeType.Guo, force=ForceType.Kolmogorov,
                              nx=n[0], ny=n[1], nz=n[2], tau=0.5005, amplitude=(1e-5, 0, 0),
                              wavelength=(n[1], 1, 1), storage=Precision.F32,
                              compute=Precision.F32, shifted=True, alpha_mode=mode)) as a:
            a.init_noise(1.0, amp, 7)
            a.iterate(40)
            out.append((a.populations(), a.alpha(), a.elbm_stats()))
    (fp, ap, sp), (fw, aw, sw) = out
    print(sp, sw, f"{(fp != fw).sum()} populations and {(ap != aw).sum()} alphas differ", flush=True)
    assert sw["learned_accepted"] > 0.05 * sw["newton"]
    assert np.array_equal(fp, fw) and np.array_equal(ap, aw)
    assert all(sp[k] == sw[k] for k in ("small", "capped", "newton", "fallback"))
