"""The first steps of an entropic handle captured in a HIP graph, with no eager step before
them: whatever such a step needs was allocated with the handle or by the choice of its mode
(an allocation would end the capture)."""
import ctypes

import numpy as np
import pytest

from metalbm_amd import AlphaMode, Algorithm, CollisionType, Config, LatticeType, Precision
from test_gpu_capture import hip

pytestmark = pytest.mark.gpu

D2Q9, D3Q27 = LatticeType.D2Q9, LatticeType.D3Q27
F64, F32 = (Precision.F64, Precision.F64, False), (Precision.F32, Precision.F32, True)

# lattice, extents, numbers, alpha mode, whether it is set on the handle or in its configuration
CASES = [
    (D3Q27, (41, 40, 42), F64, AlphaMode.WARM_RESIDUAL, True),
    (D3Q27, (41, 40, 42), F32, AlphaMode.WARM_RESIDUAL, False),
    (D3Q27, (41, 40, 42), F64, AlphaMode.NEWTON_RESIDUAL, True),
    (D2Q9, (520, 512, 1), F32, AlphaMode.WARM_RESIDUAL, False),
    (D2Q9, (64, 60, 1), F32, AlphaMode.WARM_RESIDUAL, True),
]


@pytest.mark.parametrize("c", CASES, ids=lambda c: f"{c[0].name}-{c[1][0]}-{c[2][0].name}-"
                         f"{c[3].name}-{'set' if c[4] else 'created'}")
def test_first_steps(c):
    lat, n, numbers, mode, later = c
    print("case capture first", lat.name, n, numbers[0].name, mode, later, flush=True)
    cfg = Config(lattice=lat, collision=CollisionType.ELBM, nx=n[0], ny=n[1], nz=n[2], tau=0.5005,
                 storage=numbers[0], compute=numbers[1], shifted=numbers[2],
                 alpha_mode=AlphaMode.NEWTON if later else mode)
    with Algorithm(cfg) as a, Algorithm(cfg) as b:
        for x in (a, b):
            if later:
                x.set_alpha_mode(mode)
            x.init_noise(1.0, 5e-2, 5)
            x.synchronize()
        H, P = hip(), ctypes.c_void_p
        stream, graph, run = P(), P(), P()
        assert H.hipStreamCreate(ctypes.byref(stream)) == 0
        b.set_stream(stream.value)
        assert H.hipStreamBeginCapture(stream, 1) == 0  # this thread may not allocate
        try:
            b.iterate(2)
        finally:  # a capture left open would fail the tests after this one
            ended = H.hipStreamEndCapture(stream, ctypes.byref(graph))
        assert ended == 0
        assert H.hipGraphInstantiate(ctypes.byref(run), graph, None, None,
                                     ctypes.c_size_t(0)) == 0
        for k in range(3):
            assert H.hipGraphLaunch(run, stream) == 0
            assert H.hipStreamSynchronize(stream) == 0
            a.iterate(2)
            assert np.array_equal(b.populations(), a.populations()), k
            assert np.array_equal(b.alpha(), a.alpha()), k
        b.set_stream(None)
        assert H.hipGraphExecDestroy(run) == 0 and H.hipGraphDestroy(graph) == 0
        assert H.hipStreamDestroy(stream) == 0
