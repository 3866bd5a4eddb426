"""The entropic solves of a domain of periodic copies against those of one copy, as in
tests/test_gpu_entropy_series.py, for the other number formats, sources and modes.

FP32 arithmetic: equal, the counters too.  The certified modes list cells in both
domains; the short list gives each cell a group of lanes, the long one a lane.

FP64 arithmetic: the power sums' alpha is taken wherever they decide the iterations, so
it differs from the term-by-term one by the rounding of the latter's G over |G'|: at most
2^-52 rho for the quotients under its logarithms in D2Q9, twice that in 3D; a factor of
four covers its sums and the last step's own division."""
import numpy as np
import pytest

from metalbm_amd import (AlphaMode, Algorithm, CollisionType, Config, ForceType,
                         ForcingSchemeType, LatticeType, Precision)

pytestmark = pytest.mark.gpu

D2Q9, D3Q19, D3Q27 = LatticeType.D2Q9, LatticeType.D3Q19, LatticeType.D3Q27
GUO, EDM = ForcingSchemeType.Guo, ForcingSchemeType.ExactDifferenceMethod
NEWTON, PLAIN, WARM = AlphaMode.NEWTON, AlphaMode.NEWTON_RESIDUAL, AlphaMode.WARM_RESIDUAL
F64, F32, F16 = Precision.F64, Precision.F32, Precision.F16
COPIES = {D2Q9: (8, 8, 1), D3Q19: (4, 4, 4), D3Q27: (4, 4, 4)}

# lattice, extents, storage, compute, shifted, scheme, noise, mode
CASES = [
    (D2Q9, (57, 73, 1), F64, F32, True, EDM, 6e-2, NEWTON),
    (D2Q9, (57, 73, 1), F16, F32, True, GUO, 1e-2, NEWTON),
    (D3Q27, (13, 10, 9), F16, F32, True, EDM, 5e-2, NEWTON),
    (D3Q27, (13, 10, 9), F64, F32, True, GUO, 8e-2, PLAIN),
    (D3Q19, (11, 12, 10), F32, F32, False, EDM, 5e-2, NEWTON),
    (D3Q27, (13, 10, 9), F32, F32, True, EDM, 8e-2, WARM),
    (D3Q19, (11, 12, 10), F32, F32, True, GUO, 5e-2, WARM),
    (D2Q9, (57, 73, 1), F64, F64, True, GUO, 6e-2, NEWTON),
    (D3Q27, (13, 10, 9), F64, F64, True, GUO, 5e-2, NEWTON),
    (D3Q27, (13, 10, 9), F64, F64, False, EDM, 5e-2, PLAIN),
]


def pulled(o, oc, f):
    """Pulled populations and their non-equilibrium parts, cell by cell in FP64."""
    shape, pad = (oc.nx, oc.ny, oc.nz), (0,) * (3 - oc.d)
    c = o.velocities(oc.lattice)
    fp = np.stack([np.roll(v.reshape(shape), tuple(int(x) for x in ci) + pad, (0, 1, 2)).ravel()
                   for v, ci in zip(f, c)])
    rho = fp.sum(0)
    u = c.T.astype(float) @ fp / rho
    return fp, fp - np.stack([o.equilibrium(oc, r, v) for r, v in zip(rho, u.T)], 1)


@pytest.mark.parametrize("c", CASES, ids=lambda c: f"{c[0].name}-{c[2].name}-{c[3].name}-"
                         f"{'shifted' if c[4] else 'plain'}-{c[5].name}-{c[7].name}")
def test_copies(oracle, c):
    lat, shape, storage, compute, shifted, scheme, amp, mode = c
    print("case entropic formats", lat.name, storage.name, compute.name, mode.name, flush=True)
    copies = COPIES[lat]
    large = tuple(a * b for a, b in zip(shape, copies))
    oc = oracle.Config(lattice=int(lat), collision=2, forcing_scheme=2, force=6, equilibrium=3,
                       nx=shape[0], ny=shape[1], nz=shape[2], tau=0.5005,
                       amplitude=(1e-5, 0, 0), wavelength=(shape[1], 1, 1))
    f0 = oracle.init_equilibrium(oc, np.ones(oc.cells), oracle.noise_velocity(oc, 7, amp))
    steps = 1 if compute == F64 else 3

    def tiled(v):
        return np.tile(v.reshape((-1,) + shape), (1,) + copies).reshape(v.shape[:-1] + (-1,))

    def run(n, f):
        with Algorithm(Config(lattice=lat, collision=CollisionType.ELBM, forcing_scheme=scheme,
                              force=ForceType.Kolmogorov, nx=n[0], ny=n[1], nz=n[2], tau=0.5005,
                              amplitude=(1e-5, 0, 0), wavelength=(shape[1], 1, 1),
                              storage=storage, compute=compute, shifted=shifted,
                              alpha_mode=mode)) as a:
            a.set_populations(f)
            a.iterate(steps)
            return a.populations(), a.alpha(), a.elbm_stats()
    fs, als, ss = run(shape, f0)
    fl, all_, sl = run(large, tiled(f0))
    print(f"small {ss}; large {sl}; alpha differs by {np.abs(all_ - tiled(als)).max():.2e}",
          flush=True)
    assert np.isfinite(fs).all() and ss["newton"] > 0.5 * oc.cells
    assert {k: v * int(np.prod(copies)) for k, v in ss.items()} == sl
    if compute == F32:
        np.testing.assert_array_equal(fl, tiled(fs))
        np.testing.assert_array_equal(all_, tiled(als))
        return
    # |G'| of each cell in FP64, from its pulled populations
    fp, fneq = pulled(oracle, oc, f0)
    dg = np.array([abs(oracle.entropic_dg(int(lat), fp[:, k], fneq[:, k], als[k]))
                   for k in range(oc.cells)])
    noise = (2.0 ** -52 if lat == D2Q9 else 2.0 ** -51) * fp.sum(0)
    bound = tiled(4.0 * noise / dg + 4.0 * 2.0 ** -52)
    solved = tiled(als) != 2.0
    worst = (np.abs(all_ - tiled(als)) / bound)[solved].max()
    print(f"worst {worst:.2f} of the bound", flush=True)
    assert worst <= 1.0
    np.testing.assert_array_equal(all_[~solved], 2.0)
