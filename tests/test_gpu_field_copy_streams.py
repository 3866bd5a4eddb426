"""Fields copied to the host in chunks (large requests) by a handle on streams of the
caller: the copy has to come after the steps that were enqueued just before it, also
where the stream is hipStreamPerThread, which is another stream in each host thread."""
import ctypes
import os
import threading

import numpy as np
import pytest

from metalbm_amd import Algorithm, Config, ForceType, ForcingSchemeType, LatticeType, Precision

pytestmark = pytest.mark.gpu

STREAM_PER_THREAD = 2  # hipStreamPerThread
N = (96, 80, 72)


def hip():
    for lib in ("/opt/rocm/lib/libamdhip64.so", "libamdhip64.so"):
        if os.path.sep not in lib or os.path.exists(lib):
            return ctypes.CDLL(lib)


def handle():
    a = Algorithm(Config(lattice=LatticeType.D3Q19, nx=N[0], ny=N[1], nz=N[2], tau=0.55,
                         forcing_scheme=ForcingSchemeType.Guo, force=ForceType.Sinusoidal,
                         amplitude=(1e-5, 2e-5, 1e-5), wavelength=(17.0, 9.0, 8.0),
                         storage=Precision.F64, compute=Precision.F64, shifted=False))
    a.init_noise(1.0, 2e-2, 5)
    return a


def passes(a):
    """The fields after each of three runs of steps, copied without a wait between."""
    out = []
    for _ in range(3):
        a.iterate(30, store=True)
        out.append(a.store_fields())
    return out


def same(got, want):
    return all(np.array_equal(g, w) for g3, w3 in zip(got, want) for g, w in zip(g3, w3))


@pytest.mark.parametrize("kind", ["caller", "null", "per-thread"])
def test_copy_follows_the_steps(kind):
    print("case field copy stream", kind, flush=True)
    H, stream = hip(), ctypes.c_void_p()
    with handle() as a:
        want = passes(a)
        assert sum(w.nbytes for w in want[0]) >= 8 << 20  # copied in chunks
        assert not np.array_equal(want[0][1], want[1][1])
    with handle() as a:
        if kind == "caller":
            assert H.hipStreamCreate(ctypes.byref(stream)) == 0
        a.set_stream({"caller": stream.value, "null": None, "per-thread": STREAM_PER_THREAD}[kind])
        assert same(passes(a), want)
    if stream:
        assert H.hipStreamDestroy(stream) == 0


def test_per_thread_streams_of_several_handles():
    print("case field copy per-thread streams of several handles", flush=True)
    with handle() as a:
        want = passes(a)
    got = {}

    def work(k):
        with handle() as a:
            a.set_stream(STREAM_PER_THREAD)
            got[k] = passes(a)
    threads = [threading.Thread(target=work, args=(k,)) for k in range(6)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert len(got) == 6 and all(same(g, want) for g in got.values())
