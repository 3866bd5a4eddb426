"""The two-step kernel against the one-cell-per-lane kernel.

FP64 arithmetic: the same bits (separately rounded operations in the same order).
Tolerance in FP32: a step rounds each population to FP32 after sums of at most 27 terms
on either side, so two correct kernels differ by at most 2 x 30 x 2^-24 of the
largest population a step, and BGK at tau > 1/2 near equilibrium does not amplify
it; a misplaced population is off by the noise, 1e-2 of the weights."""
import ctypes
import os

import numpy as np
import pytest

from march_cases import CASES, F64
from metalbm_amd import Algorithm, Config, KernelShape

pytestmark = pytest.mark.gpu
ULP = 2 * 30 * 2.0 ** -24


def config(c, kernel=KernelShape.AUTO):
    n = c["shape"]
    return Config(lattice=c["lattice"], nx=n[0], ny=n[1], nz=n[2], tau=0.55,
                  forcing_scheme=c["scheme"], force=c["force"], equilibrium=c["equilibrium"],
                  amplitude=(1e-5, 2e-5, -1e-5), wavelength=(n[1] / 3, 17.0, 9.0),
                  storage=c["numbers"][0], compute=c["numbers"][1], shifted=c["shifted"],
                  kernel=kernel)


def name(c):
    return (f"{c['lattice'].name}-{'x'.join(map(str, c['shape']))}-{c['scheme'].name}-"
            f"{c['force'].name}-{c['equilibrium'].name}-{'shifted' if c['shifted'] else 'plain'}-"
            f"{c['numbers'][0].name}-{c['numbers'][1].name}")


def noisy(a):
    a.init_noise(1.0, 2e-2, 5)


@pytest.mark.parametrize("c", CASES, ids=name)
def test_two_steps_per_launch(c):
    print("case march", name(c), flush=True)
    steps, out = 9, []
    for kernel in (KernelShape.AUTO, KernelShape.CELL):
        with Algorithm(config(c, kernel)) as a:
            noisy(a)
            a.iterate(steps, True)
            out.append((a.populations(), a.reduce()))
            assert a.steps_done == steps
    scale = np.abs(out[1][0]).max()
    if c["numbers"] == F64:
        assert np.array_equal(out[0][0], out[1][0])
    assert np.abs(out[0][0] - out[1][0]).max() <= steps * ULP * scale
    assert out[0][1][0] == pytest.approx(out[1][1][0], rel=steps * ULP)


def hip():
    for lib in ("/opt/rocm/lib/libamdhip64.so", "libamdhip64.so"):
        if os.path.sep not in lib or os.path.exists(lib):
            return ctypes.CDLL(lib)


def test_lattice_order_and_capture():
    """Any even number of steps ends in the lattice where it began, so replays of a
    captured graph and a pointer kept from before go on from the right populations."""
    c = CASES[0]
    print("case march capture", name(c), flush=True)
    with Algorithm(config(c)) as a, Algorithm(config(c)) as b:
        noisy(a)
        noisy(b)
        start = a.device_populations()[0]
        for n in (2, 4, 6, 8, 10):
            a.iterate(n)
            assert a.device_populations()[0] == start, n
            b.iterate(n)
        b.synchronize()
        H, P = hip(), ctypes.c_void_p
        stream, graph, run = P(), P(), P()
        assert H.hipStreamCreate(ctypes.byref(stream)) == 0
        b.set_stream(stream.value)
        assert H.hipStreamBeginCapture(stream, 2) == 0
        b.iterate(6)
        assert H.hipStreamEndCapture(stream, ctypes.byref(graph)) == 0
        assert H.hipGraphInstantiate(ctypes.byref(run), graph, None, None,
                                     ctypes.c_size_t(0)) == 0
        for _ in range(3):
            assert H.hipGraphLaunch(run, stream) == 0
            assert H.hipStreamSynchronize(stream) == 0
            a.iterate(6)
            assert np.array_equal(a.populations(), b.populations())
        b.set_stream(None)
        assert H.hipGraphExecDestroy(run) == 0 and H.hipGraphDestroy(graph) == 0
        assert H.hipStreamDestroy(stream) == 0
