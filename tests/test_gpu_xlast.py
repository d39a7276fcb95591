"""k_xlast and k4_xlast (the x faces of a 3-D stage with the update) where a wavefront's 63 cells meet the rows: rows of fewer, exactly and
more faces than a wavefront, over periodic and walled x axes and time schemes; residual, steps and a replayed run against
the oracle bit for bit, and the FP32 fluxes against the fused passes, which take the same operations."""
import numpy as np
import pytest

from cases import base_keys, smooth_state
from fenice_amd import fvg
from oracle_lib import Oracle

pytestmark = pytest.mark.gpu

WALLS = dict(bc_xmin="transmissive", bc_xmax="no_slip", bc_ymin="no_slip", bc_ymax="moving_wall", u_in="1.0")
CONFIGS = {
    "periodic-weno5-visc": (True, dict(reconstruction="weno5", use_viscous="true", mu="0.01")),
    "periodic-weno3": (True, dict(reconstruction="weno3")),
    "periodic-muscl-euler-visc": (True, dict(time_scheme="Explicit Euler", use_viscous="true", mu="0.01")),
    "walls-weno5-visc-bo1": (False, dict(WALLS, boundary_order=1, use_viscous="true", mu="0.01", reconstruction="weno5")),
    "periodic-fourth-visc": (True, dict(reconstruction="weno5", flux_quadrature="fourth", use_viscous="true", mu="0.01")),
    "walls-fourth": (False, dict(WALLS, boundary_order=2, reconstruction="weno3", flux_quadrature="fourth")),
    "walls-muscl-rk2-bo2": (False, dict(WALLS, boundary_order=2, time_scheme="SSP Runge-Kutta 2")),
}


def same(a, b):
    return np.array_equal(a.view(np.uint64), b.view(np.uint64))


@pytest.mark.parametrize("name", list(CONFIGS))
@pytest.mark.parametrize("dims", [(4, 5, 3), (61, 3, 4), (62, 4, 3), (63, 3, 5), (64, 3, 3), (127, 3, 3)])
def test_stages(name, dims):
    periodic, over = CONFIGS[name]
    keys = base_keys(*dims, periodic=periodic, **over)
    cfg = fvg.config_from_keys(keys)
    U, o = smooth_state(*dims, 9), Oracle()
    V, t = U.copy(), 0.0
    with fvg.Solver(cfg) as s:
        s.upload(U)
        R, S = s.residual()
        Ro, So = o.residual(cfg, U)
        assert S == So and same(R, Ro)
        r = s.step(t, 1e9)
        dt, S, _, ok = o.step(cfg, V, t, 1e9)
        t += dt
        assert ok and r.s_max == S and r.dt == dt and same(s.download(), V)
        tt, k, S = s.advance(t, 1e9, max_steps=5)
        for _ in range(5):
            dt, So, _, _ = o.step(cfg, V, t, 1e9)
            t += dt
        assert tt == t and S == So and same(s.download(), V)
    if "flux_quadrature" in over:   # FP64 only
        return
    outs = []
    for fused in (False, True):
        with fvg.Solver(fvg.config_from_keys(dict(keys, flux_precision="fp32"))) as s:
            s.set_fused(fused)
            s.upload(U)
            outs.append((s.advance(0.0, 1e9, max_steps=4)[0], s.download()))
    assert outs[0][0] == outs[1][0] and same(outs[0][1], outs[1][1])
