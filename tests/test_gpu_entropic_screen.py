"""The entropic step's single-precision look at a cell (largest |n| / f, smallest f)
decides only what FP64 would decide the same way: cells whose smallest population is
tiny against its weight, where f - w + w keeps no digits in FP32, and cells that are not
a number."""
import numpy as np
import pytest

from metalbm_amd import (AlphaMode, Algorithm, CollisionType, Config, ForcingSchemeType,
                         LatticeType, Precision)

pytestmark = pytest.mark.gpu

D2Q9, D3Q27 = LatticeType.D2Q9, LatticeType.D3Q27
C = np.array([(0, 0), (-1, 1), (-1, 0), (-1, -1), (1, -1), (1, 0), (1, 1), (0, -1), (0, 1)])
W = np.array([4 / 9] + [1 / 36, 1 / 9] * 4)[[0, 1, 2, 1, 1, 2, 1, 2, 2]]
THRESHOLD = 1e-3


def handle(lat, shape, numbers, mode=AlphaMode.NEWTON):
    return Algorithm(Config(
        lattice=lat, collision=CollisionType.ELBM, forcing_scheme=ForcingSchemeType.None_,
        nx=shape[0], ny=shape[1], nz=shape[2], tau=0.6, storage=numbers[0], compute=numbers[1],
        shifted=numbers[2], alpha_mode=mode))


def ma3(u):
    cu, u2 = C @ u, (u * u).sum(0)
    return W[:, None] * (1 + 3 * cu - 1.5 * u2 + 4.5 * cu ** 2 - 4.5 * cu * u2 + 4.5 * cu ** 3
                         + 1.125 * u2 ** 2 - 6.75 * cu ** 2 * u2 + 3.375 * cu ** 4)


def ratios(f):
    rho = f.sum(0)
    return np.abs(f - rho * ma3(C.T @ f / rho)) / f


def near_zero_states(n):
    """Equilibria with one population of 1e-8 to 1e-5 of its weight, that one moved off
    equilibrium by 0.6 or 1.6 times the threshold."""
    eps = np.geomspace(1e-8, 1e-5, n)
    lo, hi = np.full(n, 0.4), np.full(n, 0.7)
    for _ in range(200):  # P of the last-but-positive population falls through eps in U
        mid = 0.5 * (lo + hi)
        p = (ma3(np.stack([-mid, np.full(n, 0.05)])) / W[:, None])[4]
        lo, hi = np.where(p > eps, mid, lo), np.where(p > eps, hi, mid)
    f = ma3(np.stack([-lo, np.full(n, 0.05)]))
    f[4] *= 1 + THRESHOLD * np.where(np.arange(n) % 2, 1.6, 0.6)
    return f


def test_populations_near_zero():
    shape = (32, 32, 1)
    f = near_zero_states(shape[0] * shape[1])
    r = ratios(f)
    assert (f > 0).all()
    assert np.abs(r.max(0) / THRESHOLD - 1).min() > 0.2  # none near the threshold
    small = int((r <= THRESHOLD).all(0).sum())
    # cell x pulls population i from x - c_i
    g = np.stack([np.roll(f[i].reshape(shape[:2]), -C[i], (0, 1)).ravel() for i in range(9)])
    print("case near-zero populations", small, "of", f.shape[1], flush=True)
    with handle(D2Q9, shape, (Precision.F64, Precision.F64, True)) as a:
        a.set_populations(g)
        a.iterate(1)
        st = a.elbm_stats()
    print(st, flush=True)
    assert st["small"] == small


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
