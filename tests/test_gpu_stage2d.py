"""k_stage2d (a Runge-Kutta stage of a 2-D mesh in one launch) at the edges of its tiles: meshes of exactly one tile, one
cell more or less, several ragged tiles and thin ones, over side types, ghost slabs, viscosity and time schemes; residual,
steps and a replayed run against the oracle bit for bit, and a mesh with values out of the in-range arithmetic in some
tiles only."""
import numpy as np
import pytest

from cases import base_keys, shock_state, smooth_state
from fenice_amd import fvg
from oracle_lib import Oracle

pytestmark = pytest.mark.gpu

WALLS = dict(bc_xmin="transmissive", bc_xmax="wall", bc_ymin="no_slip", bc_ymax="moving_wall", u_in="1.0")
INOUT = dict(bc_xmin="massflow_inlet", bc_xmax="nonreflecting", bc_ymin="wall", bc_ymax="no_slip", u_in="0.5", v_in="0.1",
             rho_in="1.2", p_out="0.9")
CONFIGS = {
    "periodic-weno5": (True, dict(reconstruction="weno5")),
    "periodic-muscl-rk2-visc": (True, dict(time_scheme="SSP Runge-Kutta 2", use_viscous="true", mu="0.02")),
    "walls-muscl-visc-bo2": (False, dict(WALLS, boundary_order=2, use_viscous="true", mu="0.01")),
    "walls-weno3-visc-bo1": (False, dict(WALLS, boundary_order=1, use_viscous="true", mu="0.01", reconstruction="weno3")),
    "inout-weno5-visc-bo2": (False, dict(INOUT, boundary_order=2, use_viscous="true", mu="0.01", reconstruction="weno5")),
    "periodic-x-walls-y-euler": (False, dict(WALLS, bc_xmin="periodic", bc_xmax="periodic", boundary_order=2, time_scheme="Explicit Euler",
                                             use_viscous="true", mu="0.01")),
}


def same(a, b):
    return np.array_equal(a.view(np.uint64), b.view(np.uint64))


@pytest.mark.parametrize("name", list(CONFIGS))
@pytest.mark.parametrize("dims", [(15, 15), (16, 14), (31, 46), (2, 33), (29, 3)])
def test_stages(name, dims):
    periodic, over = CONFIGS[name]
    cfg = fvg.config_from_keys(base_keys(*dims, periodic=periodic, **over))
    U, o = smooth_state(*dims, 1, 9), Oracle()
    V, t = U.copy(), 0.0
    with fvg.Solver(cfg) as s:
        s.upload(U)
        R, S = s.residual()
        Ro, So = o.residual(cfg, U)
        assert S == So and same(R, Ro)
        for _ in range(2):
            r = s.step(t, 1e9)
            dt, S, _, ok = o.step(cfg, V, t, 1e9)
            t += dt
            assert ok and r.s_max == S and r.dt == dt and same(s.download(), V)
        tt, k, S = s.advance(t, 1e9, max_steps=6)
        for _ in range(6):
            dt, So, _, _ = o.step(cfg, V, t, 1e9)
            t += dt
        assert tt == t and S == So and same(s.download(), V)


def test_range_is_decided_per_tile():
    cfg = fvg.config_from_keys(base_keys(40, 50, reconstruction="weno5"))
    U = shock_state(40, 50, 1, 2)
    U[1000:, 2] = U[1000:, 0] * 2.0 ** -600
    o, V, t = Oracle(), U.copy(), 0.0
    with fvg.Solver(cfg) as s:
        s.upload(U)
        for _ in range(3):
            s.step(t, 1e9)
            t += o.step(cfg, V, t, 1e9)[0]
            assert same(s.download(), V)
