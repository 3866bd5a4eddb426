"""The sample log of the certified alpha modes: every solve that the correction leaves to
Newton is logged, wherever the kernels carry it out (in place or from the list of
cells), so with fraction 1 the log holds as many samples as the counters say."""
import numpy as np
import pytest

from metalbm_amd import (AlphaMode, Algorithm, CollisionType, Config, ForceType,
                         ForcingSchemeType, LatticeType, Precision)

pytestmark = pytest.mark.gpu

D2Q9, D3Q27 = LatticeType.D2Q9, LatticeType.D3Q27


@pytest.mark.parametrize("lat,shape", [(D2Q9, (57, 73, 1)), (D3Q27, (21, 20, 18)),
                                       (D3Q27, (41, 40, 42))],
                         ids=["D2Q9", "D3Q27", "D3Q27-large"])
@pytest.mark.parametrize("mode", [AlphaMode.LEARNED, AlphaMode.WARM_RESIDUAL],
                         ids=lambda m: m.name)
def test_log_holds_the_deferred_solves(lat, shape, mode):
    print(f"case sample log {lat.name} {shape} {mode.name}", flush=True)
    cfg = Config(lattice=lat, collision=CollisionType.ELBM, forcing_scheme=ForcingSchemeType.Guo,
                 force=ForceType.Kolmogorov, nx=shape[0], ny=shape[1], nz=shape[2], tau=0.5005,
                 amplitude=(1e-5, 0, 0), wavelength=(shape[1], 1, 1), storage=Precision.F32,
                 compute=Precision.F32, shifted=True, alpha_mode=mode, residual_tol=1e-13)
    with Algorithm(cfg) as a:
        a.init_noise(1.0, 5e-2, 7)
        if mode == AlphaMode.LEARNED:
            # an untrained network whose output stays within 1% of 2: starts
            # that one correction at this tolerance does not settle
            a.mlp_init(1)
            nin = a.mlp_shape()[0]
            a.set_normalization(np.zeros(nin, np.float32), np.ones(nin, np.float32), 2.0, 1e-2)
        a.sample_log_enable(4 * 3 * a.N, 1.0, 5)
        a.reset_elbm_stats()
        a.iterate(3)
        a.sample_log_disable()
        x, alpha = a.sample_log()
        st = a.elbm_stats()
    print(f"{len(alpha)} samples; {st}", flush=True)
    deferred = st["newton"] - st["learned_accepted"]
    assert deferred > 0.05 * st["newton"]
    assert len(alpha) == deferred
    assert ((alpha > 1.0) & (alpha < 2.5)).all() and np.isfinite(x).all()
