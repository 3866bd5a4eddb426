"""Configurations that take the two-step kernel: whole rows and split rows, tiles
that divide the domain and ragged ones, one range and many, a two-plane domain,
one row of tiles that is its own neighbour; each source, force axis, equilibrium
and number format."""
from metalbm_amd import (EquilibriumType, ForceType, ForcingSchemeType, LatticeType,
                         Precision)

Q19, Q27 = LatticeType.D3Q19, LatticeType.D3Q27
MA3, EXACT = EquilibriumType.TruncationMa3, EquilibriumType.Exact
NONE, GUO, EDM = (ForcingSchemeType.None_, ForcingSchemeType.Guo,
                  ForcingSchemeType.ExactDifferenceMethod)
F = ForceType


# storage, compute
F32, F64 = (Precision.F32, Precision.F32), (Precision.F64, Precision.F64)


def case(lattice, shape, scheme, force, equilibrium, shifted, numbers=F32):
    return dict(lattice=lattice, shape=shape, scheme=scheme, force=force,
                equilibrium=equilibrium, shifted=shifted, numbers=numbers)


CASES = [
    case(Q19, (70, 64, 64), GUO, F.Constant, MA3, True),
    case(Q19, (37, 211, 150), GUO, F.Kolmogorov, MA3, True),
    case(Q19, (101, 131, 97), EDM, F.Sinusoidal, MA3, True),
    case(Q19, (2, 401, 600), NONE, F.None_, MA3, False),
    case(Q19, (61, 9, 1100), GUO, F.Sinusoidal, MA3, False),
    case(Q27, (97, 161, 129), GUO, F.Kolmogorov, EXACT, True),
    case(Q27, (129, 127, 127), EDM, F.Constant, EXACT, False),
    case(Q27, (29, 70, 530), EDM, F.Sinusoidal, MA3, True),
    case(Q27, (512, 32, 33), NONE, F.None_, EXACT, True),
    case(Q19, (71, 90, 77), GUO, F.Kolmogorov, MA3, False, F64),
    case(Q19, (90, 70, 301), EDM, F.Sinusoidal, MA3, False, F64),
    case(Q19, (82, 81, 64), GUO, F.Constant, MA3, True, F64),
    case(Q27, (57, 255, 129), NONE, F.None_, MA3, False, F64),
]


def kernel_of(c):
    """Columns, interior columns, force table entries, values to a line and cost limit
    of the two-step kernel."""
    q27, exact = c["lattice"] == Q27, c["equilibrium"] == EXACT
    source, fp64 = c["scheme"] != NONE, c["numbers"] == F64
    side = 264 if source and c["force"] in (F.Kolmogorov, F.Sinusoidal) else 0
    limit = (4.9 if fp64 else 3.9 if exact and source else 6.1 if q27 else
             5.3 if c["scheme"] == EDM else 13.0)
    size = 8 if fp64 else 4
    lds = 163840 - 3 * side * size
    interior = 512 if fp64 else 1024 if q27 else 2048
    return lds // ((24 if q27 else 16) * size) // 4 * 4, interior, side, 128 // size, limit
