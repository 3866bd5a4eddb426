"""Single-precision results do not depend on how steps are split over calls, on which of
them store, nor on the kernel shape: all kernels that a configuration may run share one
collision, rounded the same way, so every comparison is for equality.  And with the
polynomial equilibrium that collision keeps the mass: its roundings have no preferred
sign."""
import numpy as np
import pytest

from metalbm_amd import (Algorithm, Config, EquilibriumType, ForceType, ForcingSchemeType,
                         KernelShape, LatticeType, Precision)

pytestmark = pytest.mark.gpu

D2Q9, Q19, Q27 = LatticeType.D2Q9, LatticeType.D3Q19, LatticeType.D3Q27
MA3, EXACT = EquilibriumType.TruncationMa3, EquilibriumType.Exact
NONE, GUO, EDM = (ForcingSchemeType.None_, ForcingSchemeType.Guo,
                  ForcingSchemeType.ExactDifferenceMethod)
F = ForceType

# lattice, extents, scheme, force, equilibrium, storage, shifted, cells per lane of the
# vector kernel (0: none for this extent)
CASES = [
    (Q19, (70, 64, 64), GUO, F.Constant, MA3, "F32", True, 4),
    (Q19, (101, 131, 98), EDM, F.Kolmogorov, MA3, "F32", True, 2),
    (Q19, (61, 90, 101), NONE, F.None_, MA3, "F32", False, 0),
    (Q27, (160, 128, 100), GUO, F.Sinusoidal, EXACT, "F32", True, 4),
    (Q27, (127, 128, 126), EDM, F.Constant, EXACT, "F32", False, 2),
    (Q27, (97, 161, 129), GUO, F.Kolmogorov, EXACT, "F32", True, 0),
    (Q27, (29, 70, 530), EDM, F.Sinusoidal, MA3, "F32", True, 2),
    (Q27, (129, 127, 128), GUO, F.Constant, MA3, "F32", False, 4),
    (Q27, (512, 32, 33), NONE, F.None_, EXACT, "F32", True, 0),
    (D2Q9, (131, 124), GUO, F.Kolmogorov, MA3, "F32", True, 4),
    (D2Q9, (300, 290), EDM, F.Sinusoidal, MA3, "F32", False, 2),
    (D2Q9, (40, 37), EDM, F.Kolmogorov, EXACT, "F32", True, 0),
    (D2Q9, (300, 12), GUO, F.Sinusoidal, EXACT, "F32", True, 4),
    # FP16's vector kernel is left out: it converts two results at once, after they
    # were rounded, where the others round a fused operation's result to FP16 directly
    (D2Q9, (257, 301), GUO, F.Kolmogorov, MA3, "F16", True, 0),
    (D2Q9, (1030, 704), NONE, F.None_, MA3, "F16", True, 0),
    (D2Q9, (400, 333), EDM, F.Sinusoidal, MA3, "F16", True, 0),
    (D2Q9, (40, 36), GUO, F.Constant, EXACT, "F16", True, 0),
    (D2Q9, (45, 38), EDM, F.Sinusoidal, EXACT, "F16", True, 0),
    (D2Q9, (150, 90), NONE, F.None_, EXACT, "F16", True, 0),
]
# twelve steps: (steps, whether the last one stores)
SPLITS = [[(12, True)], [(1, False)] * 11 + [(1, True)], [(5, True), (7, True)],
          [(8, False), (4, True)], [(3, False), (2, True), (6, False), (1, True)]]


def config(c, kernel):
    lat, n, scheme, force, equilibrium, storage, shifted, _ = c
    return Config(lattice=lat, nx=n[0], ny=n[1], nz=n[2] if len(n) > 2 else 1, tau=0.55,
                  forcing_scheme=scheme, force=force, equilibrium=equilibrium,
                  amplitude=(1e-5, 2e-5, -1e-5), wavelength=(n[1] / 3, 17.0, 9.0),
                  storage=Precision[storage], compute=Precision.F32, shifted=shifted,
                  kernel=kernel)


@pytest.mark.parametrize("c", CASES, ids=lambda c: f"{c[0].name}-{'x'.join(map(str, c[1]))}-"
                         f"{c[2].name}-{c[3].name}-{c[4].name}-{c[5]}")
def test_any_split_and_shape(c):
    print("case call split", c[0].name, c[1], flush=True)
    shapes = [KernelShape.AUTO, KernelShape.CELL] + ([KernelShape.VECTOR] if c[7] else [])
    out = []
    for kernel in shapes:
        for split in SPLITS if kernel == KernelShape.AUTO else SPLITS[:1]:
            with Algorithm(config(c, kernel)) as a:
                a.init_noise(1.0, 2e-2, 5)
                for steps, store in split:
                    a.iterate(steps, store=store)
                out.append((kernel.name, split, (a.populations(),) + a.store_fields()))
    for name, split, got in out[1:]:
        for k, (g, w) in enumerate(zip(got, out[0][2])):
            assert np.array_equal(g, w), (name, split, k, np.abs(g - w).max())


@pytest.mark.parametrize("scheme", [NONE, GUO, EDM], ids=lambda s: s.name)
def test_mass_does_not_drift(scheme):
    """Noise of 1e-2 leaves populations of 3e-3 or less, rounded to 2^-34 of 1 (standard
    deviation 7e-11 for each of nine); over 96 x 96 cells and 2000 independent steps the
    mean density then moves by 1e-10, and 6e-10 is six times that."""
    print("case mass", scheme.name, flush=True)
    c = (D2Q9, (96, 96), scheme, F.Constant if scheme != NONE else F.None_, MA3, "F32", True,
         0)
    cfg = config(c, KernelShape.AUTO)
    cfg.tau, cfg.amplitude = 0.53, (1e-6, 5e-7, 0.0)
    with Algorithm(cfg) as a:
        a.init_noise(1.0, 1e-2, 42)
        before = a.populations().sum()
        a.iterate(2000)
        drift = (a.populations().sum() - before) / a.N
    print(f"mean density moved by {drift:.2e}", flush=True)
    assert abs(drift) <= 6e-10
