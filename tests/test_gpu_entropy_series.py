"""The entropic solve from power sums against the term-by-term solve.

A domain of many periodic copies of a small one holds the same cells; the
small domain takes the term-by-term kernels and the large one the power sums
with their list of cells, so every copy must end with the small domain's
populations.  The two solvers round alpha differently (1e-10 to 1e-13), but
where that could change the relaxation rate as it is stored and applied, or
the iteration count, the series leaves the cell to the other solver: the
populations, the stored alpha and the counters are compared exactly."""
import sys

import numpy as np
import pytest

from metalbm_amd import (AlphaMode, Algorithm, CollisionType, Config, ForceType,
                         ForcingSchemeType, LatticeType, Precision)

pytestmark = pytest.mark.gpu

D2Q9, D3Q19, D3Q27 = LatticeType.D2Q9, LatticeType.D3Q19, LatticeType.D3Q27

# (lattice, extents, copies per axis, noise, mode): weak noise near equilibrium
# (every cell within the short series), strong noise (the stored-alpha centre,
# cells out of reach, capped cells); ragged rows and partial workgroups.
CASES = [
    (D2Q9, (57, 73, 1), (8, 8, 1), 1e-3, AlphaMode.NEWTON),
    (D2Q9, (64, 64, 1), (8, 8, 1), 6e-2, AlphaMode.NEWTON),
    (D3Q27, (13, 10, 9), (4, 4, 4), 1e-2, AlphaMode.NEWTON),
    (D3Q27, (13, 10, 9), (4, 4, 4), 8e-2, AlphaMode.NEWTON),
    (D3Q27, (8, 8, 16), (4, 4, 4), 8e-2, AlphaMode.NEWTON_RESIDUAL),
    (D3Q19, (11, 12, 10), (4, 4, 4), 5e-2, AlphaMode.NEWTON),
    (D3Q19, (11, 12, 10), (4, 4, 4), 5e-2, AlphaMode.NEWTON_RESIDUAL),
]


@pytest.mark.parametrize("lat,shape,copies,amp,mode", CASES,
                         ids=[f"{c[0].name}-{c[4].name}-{c[3]:g}" for c in CASES])
@pytest.mark.parametrize("spread", [False, True], ids=["warm", "spread"])
def test_series_matches_termwise(oracle, lat, shape, copies, amp, mode, spread):
    def config(n):
        return Config(lattice=lat, collision=CollisionType.ELBM,
                      forcing_scheme=ForcingSchemeType.Guo, force=ForceType.Kolmogorov,
                      nx=n[0], ny=n[1], nz=n[2], tau=0.5005, amplitude=(1e-5, 0, 0),
                      wavelength=(shape[1], 1, 1), storage=Precision.F32, compute=Precision.F32,
                      shifted=True, alpha_mode=mode)
    print(f"case series {lat.name} {shape} x {copies} {mode.name} spread={spread}", flush=True)
    sys.stdout.flush()
    large = tuple(a * b for a, b in zip(shape, copies))
    small_cells, large_cells = int(np.prod(shape)), int(np.prod(large))
    assert small_cells < 1 << 16 and large_cells >= (1 << 18 if lat == D2Q9 else 1 << 16)
    cfg = config(shape)
    oc = oracle.Config(lattice=int(lat), collision=2, forcing_scheme=2, force=6, equilibrium=3,
                       nx=shape[0], ny=shape[1], nz=shape[2], tau=0.5005,
                       amplitude=(1e-5, 0, 0), wavelength=(shape[1], 1, 1))
    f0 = oracle.init_equilibrium(oc, np.ones(oc.cells), oracle.noise_velocity(oc, 7, amp))
    alpha0 = np.full(oc.cells, 2.0)
    if spread:  # starts on both sides of the root and of G's maximum
        alpha0 = np.random.default_rng(3).uniform(0.3, 2.5, oc.cells)

    def tiled(v):
        return np.tile(v.reshape((-1,) + shape), (1,) + copies).reshape(v.shape[:-1] + (-1,))

    def run(c, f, al):
        with Algorithm(c) as a:
            a.set_populations(f)
            a.set_alpha(al)
            a.iterate(3)
            return a.populations(), a.alpha(), a.elbm_stats()
    fs, als, ss = run(cfg, f0, alpha0)
    fl, all_, sl = run(config(large), tiled(f0), tiled(alpha0))
    copies_n = large_cells // small_cells
    print(f"small {ss}; large {sl}", flush=True)
    assert np.isfinite(fs).all()
    np.testing.assert_array_equal(fl, tiled(fs))
    np.testing.assert_array_equal(all_, tiled(als))
    assert {k: v * copies_n for k, v in ss.items()} == sl
