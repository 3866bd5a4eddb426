"""Fields copied to the host in chunks by several threads (large requests) against the
same fields asked for one by one (small requests: one copy each)."""
import ctypes
import threading

import numpy as np
import pytest

from metalbm_amd import Algorithm, Config, ForceType, ForcingSchemeType, LatticeType, Precision
from metalbm_amd.capi import lib

pytestmark = pytest.mark.gpu

RING = 8 << 20  # requests of fewer bytes are copied directly

# just over the limit with ragged chunks, whole chunks, 2D
SHAPES = [(LatticeType.D3Q19, (53, 51, 52)), (LatticeType.D3Q19, (64, 64, 32)),
          (LatticeType.D2Q9, (431, 433, 1))]


def handle(lat, n):
    a = Algorithm(Config(lattice=lat, nx=n[0], ny=n[1], nz=n[2], tau=0.55,
                         forcing_scheme=ForcingSchemeType.Guo, force=ForceType.Sinusoidal,
                         amplitude=(1e-5, 2e-5, 1e-5), wavelength=(17.0, 9.0, 8.0),
                         storage=Precision.F64, compute=Precision.F64, shifted=False))
    a.init_noise(1.0, 2e-2, 5)
    a.iterate(3, store=True)
    return a


def one_by_one(a):
    parts = []
    for k, shape in enumerate([(a.N,), (a.D, a.N), (a.N,), (a.D, a.N)]):
        out = np.empty(shape)
        assert out.nbytes < RING
        args = [None] * 4
        args[k] = out.ctypes.data_as(ctypes.POINTER(ctypes.c_double))
        assert lib().lbm_get_fields(a._h, *args) == 0
        parts.append(out)
    return parts


@pytest.mark.parametrize("lat,n", SHAPES, ids=[f"{s[0].name}-{s[1][0]}" for s in SHAPES])
def test_chunks_match_direct_copies(lat, n):
    print("case field copy", lat.name, n, flush=True)
    with handle(lat, n) as a, handle(lat, n) as b:
        want = one_by_one(a)
        assert sum(w.nbytes for w in want) >= RING
        got = {}
        threads = [threading.Thread(target=lambda k=k, x=x: got.__setitem__(
            k, [x.store_fields() for _ in range(3)])) for k, x in (("a", a), ("b", b))]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
    for results in got.values():
        for r in results:
            for g, w in zip(r, want):
                assert np.array_equal(g, w)
    assert len(got) == 2
