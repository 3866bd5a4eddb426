"""The fields that the vector kernel stores, a lane's V cells at a time, against the
one-cell kernel's: moments of the same populations by the same operations, so equal.  Rows of
one segment of 64 V cells, of several, and with a part of one at the end."""
import numpy as np
import pytest

from metalbm_amd import (Algorithm, Config, ForceType, ForcingSchemeType, KernelShape,
                         LatticeType, Precision)

pytestmark = pytest.mark.gpu

D2Q9, Q19, Q27 = LatticeType.D2Q9, LatticeType.D3Q19, LatticeType.D3Q27
NONE, GUO, EDM = (ForcingSchemeType.None_, ForcingSchemeType.Guo,
                  ForcingSchemeType.ExactDifferenceMethod)

CASES = [  # lattice, extents, scheme, force, storage
    (D2Q9, (9, 1032, 1), GUO, ForceType.Sinusoidal, "F16"),
    (D2Q9, (33, 516, 1), EDM, ForceType.Kolmogorov, "F16"),
    (D2Q9, (20, 130, 1), NONE, ForceType.None_, "F16"),
    (D2Q9, (30, 516, 1), NONE, ForceType.Kolmogorov, "F32"),
    (D2Q9, (30, 130, 1), GUO, ForceType.Sinusoidal, "F32"),
    (Q19, (5, 7, 264), EDM, ForceType.Sinusoidal, "F32"),
    (Q19, (6, 5, 34), NONE, ForceType.None_, "F32"),
    (Q27, (5, 6, 16), GUO, ForceType.Kolmogorov, "F32"),
]


@pytest.mark.parametrize("c", CASES, ids=lambda c: f"{c[0].name}-{c[1][-1 if c[1][2] > 1 else 1]}"
                         f"-{c[2].name}-{c[4]}")
def test_fields(c):
    lat, n, scheme, force, storage = c
    print("case vector fields", lat.name, n, scheme.name, storage, flush=True)
    out = []
    for kernel in (KernelShape.CELL, KernelShape.VECTOR):
        cfg = Config(lattice=lat, nx=n[0], ny=n[1], nz=n[2], tau=0.6, forcing_scheme=scheme,
                     force=force, amplitude=(1e-4, 2e-4, -1e-4), wavelength=(n[1], 17.0, 9.0),
                     storage=Precision[storage], compute=Precision.F32, shifted=True,
                     kernel=kernel)
        with Algorithm(cfg) as a:
            a.init_noise(1.0, 2e-2, 7)
            a.iterate(1, store=True)
            out.append(a.store_fields())
    for k, (got, want) in enumerate(zip(*out)):
        assert np.array_equal(got, want), (k, np.abs(got - want).max())
