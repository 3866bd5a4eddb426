"""The multi-step 2D kernel against the one-cell-per-lane kernel: each width of tile,
whole and split axes, ragged remainders, domains thinner than the halo, every count of
steps up to two launches, stored fields, forces along x, along y and per cell.

FP64 keeps every bit.  FP32: a step rounds each population after sums of at most nine
terms, so two correct kernels differ by at most 2 x 15 x 2^-24 of the largest
population a step, and BGK at tau > 1/2 near equilibrium does not amplify it.  FP16: the
same with a rounding to 2^-11 of a population's weight, which an FP32 difference can
tip."""
import numpy as np
import pytest

from metalbm_amd import (Algorithm, Config, EquilibriumType, ForceType, ForcingSchemeType,
                         KernelShape, LatticeType, Precision)

pytestmark = pytest.mark.gpu

MA3, EXACT = EquilibriumType.TruncationMa3, EquilibriumType.Exact
NONE, GUO, EDM = (ForcingSchemeType.None_, ForcingSchemeType.Guo,
                  ForcingSchemeType.ExactDifferenceMethod)
F = ForceType
F64, F32, F16 = ((Precision.F64, Precision.F64, False, 0.0),
                 (Precision.F32, Precision.F32, True, 2 * 15 * 2.0 ** -24),
                 (Precision.F16, Precision.F32, True, 2 * 2.0 ** -11))

CASES = [
    ((32, 32), GUO, F.Kolmogorov, MA3, F64), ((33, 47), EDM, F.Sinusoidal, EXACT, F64),
    ((131, 125), GUO, F.Constant, MA3, F32), ((190, 203), NONE, F.None_, MA3, F64),
    ((3, 300), GUO, F.Sinusoidal, MA3, F64), ((300, 12), GUO, F.Kolmogorov, EXACT, F32),
    ((300, 290), EDM, F.Sinusoidal, MA3, F32), ((511, 520), GUO, F.Kolmogorov, MA3, F64),
    ((1000, 60), GUO, F.Sinusoidal, MA3, F64), ((2, 2000), GUO, F.Constant, MA3, F32),
    ((1023, 777), NONE, F.None_, MA3, F32), ((257, 301), GUO, F.Kolmogorov, MA3, F16),
    ((40, 37), EDM, F.Kolmogorov, EXACT, F16), ((1030, 701), GUO, F.Sinusoidal, MA3, F16),
]


def config(shape, scheme, force, equilibrium, numbers, kernel):
    return Config(lattice=LatticeType.D2Q9, nx=shape[0], ny=shape[1], nz=1, tau=0.55,
                  forcing_scheme=scheme, force=force, equilibrium=equilibrium,
                  amplitude=(1e-5, 2e-5, 0.0), wavelength=(shape[1] / 3, 17.0, 1.0),
                  force_kmin=2, force_kmax=4, storage=numbers[0], compute=numbers[1],
                  shifted=numbers[2], kernel=kernel)


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"{c[0][0]}x{c[0][1]}-{c[1].name}-"
                         f"{c[2].name}-{c[3].name}-{c[4][0].name}")
def test_several_steps_per_launch(case):
    print("case tile", case[0], flush=True)
    numbers, total = case[4], 0
    with Algorithm(config(*case, KernelShape.AUTO)) as a, \
            Algorithm(config(*case, KernelShape.CELL)) as b:
        for x in (a, b):
            x.init_noise(1.0, 2e-2, 5)
        for steps in (1, 2, 3, 4, 5, 6, 9, 10):
            total += steps
            for x in (a, b):
                x.iterate(steps, store=steps % 3 == 0)
        start = a.device_populations()[0]
        a.iterate(8)
        assert a.device_populations()[0] == start
        a.iterate(3, store=True)
        b.iterate(11, store=True)
        total += 11
        got, want = (a.populations(),) + a.store_fields(), (b.populations(),) + b.store_fields()
        assert a.steps_done == b.steps_done == total
    for g, w in zip(got, want):
        if numbers is F64:
            assert np.array_equal(g, w)
        assert np.abs(g - w).max() <= total * numbers[3] * max(np.abs(w).max(), 1e-30)


@pytest.mark.parametrize("shape", [(64, 96), (300, 290)])
def test_force_field(shape):
    """A force per cell, rebuilt from the fields that the last call stored."""
    print("case tile force field", shape, flush=True)
    out = []
    for kernel in (KernelShape.AUTO, KernelShape.CELL):
        with Algorithm(config(shape, EDM, F.Turbulent2D, MA3, F32, kernel)) as a:
            a.init_noise(1.0, 2e-2, 5)
            for steps in (5, 10, 4):
                a.iterate(steps, store=True)
            out.append((a.populations(),) + a.store_fields())
    for g, w in zip(*out):
        assert np.abs(g - w).max() <= 19 * F32[3] * max(np.abs(w).max(), 1e-30)
