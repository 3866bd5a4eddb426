"""Pinned memory for copying fields is shared by the handles of a process: copying from
many handles, one after another or at once, takes that of a few."""
import ctypes
import threading

import numpy as np
import pytest

from metalbm_amd import Algorithm, Config, LatticeType
from metalbm_amd.capi import lib

pytestmark = pytest.mark.gpu

N, HANDLES = (64, 64, 64), 24
RING = 8 << 20  # bytes of one set of pinned chunks


def mapped():
    """Bytes of address space in use (pinned memory is mapped, not counted as resident)."""
    with open("/proc/self/statm") as f:
        return int(f.read().split()[0]) * 4096


def copy(a, out):
    args = [o.ctypes.data_as(ctypes.POINTER(ctypes.c_double)) for o in out]
    assert lib().lbm_get_fields(a._h, *args) == 0


def buffers(a):
    return [np.zeros((a.N,)), np.zeros((a.D, a.N)), np.zeros((a.N,)), np.zeros((a.D, a.N))]


def test_handles_share_the_pinned_memory():
    print("case pinned memory", flush=True)
    handles = []
    try:
        for k in range(HANDLES):
            handles.append(Algorithm(Config(lattice=LatticeType.D3Q19, nx=N[0], ny=N[1], nz=N[2])))
            handles[-1].init_noise(1.0, 1e-2, k)
            handles[-1].iterate(2, store=True)
            handles[-1].synchronize()
        out = buffers(handles[0])
        copy(handles[0], out)  # the first copy's threads and stream
        start = mapped()
        for a in handles[1:]:
            copy(a, out)
        grown = mapped() - start
        print(f"{grown / 2 ** 20:.1f} MiB for {HANDLES - 1} more handles", flush=True)
        assert grown < (HANDLES - 1) * RING // 4
        # all at once: each gets its own handle's fields
        got = {}
        threads = [threading.Thread(target=lambda k=k, a=a: got.__setitem__(k, a.store_fields()))
                   for k, a in enumerate(handles)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert len(got) == HANDLES
        for k, a in enumerate(handles):
            copy(a, out)
            for g, w in zip(got[k], out):
                assert np.array_equal(g.reshape(w.shape), w), k
    finally:
        for a in handles:
            a.close()
