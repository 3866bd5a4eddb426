"""Configurations that take the two-step kernel: whole rows and split rows, tiles
that divide the domain and ragged ones, one range and many, a two-plane domain,
one row of tiles that is its own neighbour; each source, force axis, equilibrium
and number format."""
from metalbm_amd import EquilibriumType, ForceType, ForcingSchemeType, LatticeType

Q19, Q27 = LatticeType.D3Q19, LatticeType.D3Q27
MA3, EXACT = EquilibriumType.TruncationMa3, EquilibriumType.Exact
NONE, GUO, EDM = (ForcingSchemeType.None_, ForcingSchemeType.Guo,
                  ForcingSchemeType.ExactDifferenceMethod)
F = ForceType


def case(lattice, shape, scheme, force, equilibrium, shifted):
    return dict(lattice=lattice, shape=shape, scheme=scheme, force=force,
                equilibrium=equilibrium, shifted=shifted)


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
]


def kernel_of(c):
    """(kernel index, limit) of tests/native/march_rules.cpp."""
    q27, exact = c["lattice"] == Q27, c["equilibrium"] == EXACT
    source = c["scheme"] != NONE
    side = source and c["force"] in (F.Kolmogorov, F.Sinusoidal)
    limit = 3.9 if exact and source else 6.1 if q27 else 5.3 if c["scheme"] == EDM else 13.0
    return 2 * q27 + side, limit
