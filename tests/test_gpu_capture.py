"""Steps captured in a HIP graph and replayed against the same steps taken eagerly: the
several-step 2D kernel, and the entropic step with its list of cells (counters that
alternate from step to step, cleared by a kernel at the start of each call)."""
import ctypes
import os

import numpy as np
import pytest

from metalbm_amd import (AlphaMode, Algorithm, CollisionType, Config, ForceType,
                         ForcingSchemeType, LatticeType, Precision)

pytestmark = pytest.mark.gpu

D2Q9, D3Q27 = LatticeType.D2Q9, LatticeType.D3Q27
F64, F32, F16 = ((Precision.F64, Precision.F64, False), (Precision.F32, Precision.F32, True),
                 (Precision.F16, Precision.F32, True))

# lattice, extents, numbers, alpha mode (None: BGK), noise, steps of the captured call
CASES = [
    (D2Q9, (128, 128, 1), F64, None, 2e-2, 10),
    (D2Q9, (300, 290, 1), F32, None, 2e-2, 4),
    (D2Q9, (257, 301, 1), F16, None, 2e-2, 6),
    (D2Q9, (520, 512, 1), F32, AlphaMode.NEWTON, 6e-2, 2),
    (D3Q27, (41, 40, 42), F32, AlphaMode.NEWTON, 5e-2, 4),
    (D3Q27, (41, 40, 42), F32, AlphaMode.NEWTON_RESIDUAL, 5e-2, 2),
    (D3Q27, (21, 20, 18), F32, AlphaMode.WARM_RESIDUAL, 5e-2, 2),
]


def hip():
    for lib in ("/opt/rocm/lib/libamdhip64.so", "libamdhip64.so"):
        if os.path.sep not in lib or os.path.exists(lib):
            return ctypes.CDLL(lib)


@pytest.mark.parametrize("c", CASES, ids=lambda c: f"{c[0].name}-{c[1][0]}-{c[2][0].name}-"
                         f"{c[3].name if c[3] is not None else 'BGK'}")
def test_replays(c):
    lat, n, numbers, mode, amp, steps = c
    print("case capture", lat.name, n, numbers[0].name, mode, flush=True)
    cfg = Config(lattice=lat, collision=CollisionType.BGK if mode is None else CollisionType.ELBM,
                 forcing_scheme=ForcingSchemeType.Guo, force=ForceType.Kolmogorov, nx=n[0],
                 ny=n[1], nz=n[2], tau=0.55 if mode is None else 0.5005, amplitude=(1e-5, 0, 0),
                 wavelength=(n[1], 1, 1), storage=numbers[0], compute=numbers[1],
                 shifted=numbers[2], alpha_mode=mode or AlphaMode.NEWTON)

    def state(a):
        out = (a.populations(),) + a.store_fields()
        if mode is None:
            return out, None
        return out + (a.alpha(),), a.elbm_stats()

    with Algorithm(cfg) as a, Algorithm(cfg) as b:
        for x in (a, b):
            x.init_noise(1.0, amp, 5)
            x.iterate(steps, store=True)
            x.synchronize()
        H, P = hip(), ctypes.c_void_p
        stream, graph, run = P(), P(), P()
        assert H.hipStreamCreate(ctypes.byref(stream)) == 0
        b.set_stream(stream.value)
        assert H.hipStreamBeginCapture(stream, 2) == 0
        b.iterate(steps, store=True)
        assert H.hipStreamEndCapture(stream, ctypes.byref(graph)) == 0
        assert H.hipGraphInstantiate(ctypes.byref(run), graph, None, None,
                                     ctypes.c_size_t(0)) == 0
        for k in range(4):
            assert H.hipGraphLaunch(run, stream) == 0
            assert H.hipStreamSynchronize(stream) == 0
            if k == 2:  # an eager call between two replays
                b.iterate(steps, store=True)
                a.iterate(steps, store=True)
            a.iterate(steps, store=True)
            (got, gs), (want, ws) = state(b), state(a)
            for g, w in zip(got, want):
                assert np.array_equal(g, w), k
            assert gs == ws
        b.set_stream(None)
        assert H.hipGraphExecDestroy(run) == 0 and H.hipGraphDestroy(graph) == 0
        assert H.hipStreamDestroy(stream) == 0
