"""A handle's configuration names the kernel that was asked for: a handle created from it
is the same kind of handle, with the automatic choice where that was the first one's."""
import ctypes

import numpy as np
import pytest

from metalbm_amd import Algorithm, Config, KernelShape, LatticeType, Precision, kernel_shape
from metalbm_amd.capi import lib

pytestmark = pytest.mark.gpu

CASES = [(LatticeType.D2Q9, (128, 128, 1), "F64", False), (LatticeType.D3Q19, (64, 64, 64), "F32", True)]


@pytest.mark.parametrize("kernel", [KernelShape.AUTO, KernelShape.CELL, KernelShape.VECTOR],
                         ids=lambda k: k.name)
@pytest.mark.parametrize("case", CASES, ids=lambda c: c[0].name)
def test_round_trip(case, kernel):
    print("case handle config", case[0].name, kernel.name, flush=True)
    lat, n, storage, shifted = case
    cfg = Config(lattice=lat, nx=n[0], ny=n[1], nz=n[2], tau=0.55, storage=Precision[storage],
                 compute=Precision[storage], shifted=shifted, kernel=kernel)
    with Algorithm(cfg) as a:
        c = a.handle_config()
        assert c.kernel == int(kernel)
        assert bytes(c) == bytes(cfg.to_c())
        if kernel != KernelShape.AUTO:
            assert kernel_shape(cfg)[0] == kernel
        a.init_noise(1.0, 1e-3, 3)
        a.iterate(8)
        again = ctypes.c_void_p()
        assert lib().lbm_create(ctypes.byref(c), ctypes.byref(again)) == 0
        try:
            assert lib().lbm_init_noise(again, 1.0, 1e-3, 3) == 0
            assert lib().lbm_step(again, 8, 0) == 0
            f = np.empty((a.Q, a.N))
            p = f.ctypes.data_as(ctypes.POINTER(ctypes.c_double))
            assert lib().lbm_get_populations(again, p) == 0
            assert np.array_equal(f, a.populations())
        finally:
            lib().lbm_destroy(again)
