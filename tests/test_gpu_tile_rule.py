"""Which 2-D meshes run by tiles (k_stage2d, k_hancock_step2d) and which by the separate passes: long meshes of few rows
take the latter, from the first mesh of more than 1,024 tiles on, and both give the oracle's bits."""
import numpy as np
import pytest

from cases import base_keys, smooth_state
from fenice_amd import fvg
from oracle_lib import Oracle

pytestmark = pytest.mark.gpu

ROW = dict(bc_xmin="transmissive", bc_xmax="wall", bc_ymin="periodic", bc_ymax="periodic")
HANCOCK = dict(time_scheme="MUSCL-Hancock")


@pytest.mark.parametrize("dims,over,tiles", [
    ((15360, 1), dict(periodic=False, reconstruction="weno5", **ROW), True),
    ((15361, 1), dict(periodic=False, reconstruction="weno5", **ROW), False),
    ((15361, 10), dict(use_viscous="true", mu="0.01", time_scheme="SSP Runge-Kutta 2"), False),
    ((15361, 10), dict(time_scheme="Explicit Euler"), True),
    ((15361, 11), dict(use_viscous="true", mu="0.01", time_scheme="SSP Runge-Kutta 2"), True),
    ((7681, 17), dict(), False), ((5200, 31), dict(reconstruction="weno3"), True), ((3, 15500), dict(), True),
    ((14336, 9), HANCOCK, True), ((14337, 9), HANCOCK, False), ((14337, 10), HANCOCK, True), ((7169, 15), HANCOCK, False)])
def test_route_and_bits(dims, over, tiles):
    cfg = fvg.config_from_keys(base_keys(*dims, **over))
    U, o = smooth_state(*dims, 1, 9), Oracle()
    V, t, lag = U.copy(), 0.0, 0.0
    with fvg.Solver(cfg) as s:
        s.upload(U)
        s.set_timing(True)
        for _ in range(2):
            r = s.step(t, 1e9)
            dt, S, lag, ok = o.step(cfg, V, t, 1e9, 0.0, lag)
            t += dt
            assert ok and r.dt == dt and r.s_max == S
        assert np.array_equal(s.download().view(np.uint64), V.view(np.uint64))
        k = s.kernel_times()
        assert ((k["k_faces_y"][1] == 0) if cfg.time_scheme != 3 else (k["k_cells"][1] <= 1)) == tiles
