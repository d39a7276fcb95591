"""3-D contexts hold planes of x-face fluxes only where a pass stores them: a Runge-Kutta run does without, a residual
with a predictor half step makes them, and runs go on as before on either side of it."""
import ctypes as C

import numpy as np
import pytest

from cases import base_keys, smooth_state
from fenice_amd import fvg
from oracle_lib import Oracle

pytestmark = pytest.mark.gpu

WALLS = dict(bc_xmin="wall", bc_xmax="transmissive", bc_ymin="no_slip", bc_ymax="wall", bc_zmin="periodic", bc_zmax="periodic")


def same(a, b):
    return np.array_equal(a.view(np.uint64), b.view(np.uint64))


def free_bytes():
    hip = C.CDLL("libamdhip64.so")
    free, total = C.c_size_t(), C.c_size_t()
    assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


def test_runge_kutta_context_has_no_x_planes():
    n = 128
    fvg.Solver(fvg.config_from_keys(base_keys(4, 4, 4))).close()   # the device is up
    before = free_bytes()
    with fvg.Solver(fvg.config_from_keys(base_keys(n, n, n, reconstruction="weno5", use_viscous="true", mu="0.01"))) as s:
        used = before - free_bytes()
        cells, padded, face = n ** 3, (n + 64) * (n + 6) ** 2, n * n * (n + 1)
        assert used <= 8 * (3 * 5 * cells + 5 * padded + 9 * cells + 2 * 9 * face) + (64 << 20), used   # U, Ut, Rb; W; G; y and z
        s.upload(smooth_state(n, n, n, 1))
        s.residual(1e-3)
        assert before - free_bytes() >= used + 8 * 9 * face   # and the predicted states


@pytest.mark.parametrize("over", [dict(use_viscous="true", mu="0.01"), dict(periodic=False, boundary_order=2, **WALLS),
                                  dict(time_scheme="Explicit Euler"), dict(reconstruction="none", time_scheme="Explicit Euler"),
                                  dict(time_scheme="MUSCL-Hancock")])
def test_predictor_residual_between_steps(over):
    dims = (9, 8, 7)
    cfg = fvg.config_from_keys(base_keys(*dims, **over))
    U, o, t, lag = smooth_state(*dims, 9), Oracle(), 0.0, 0.0
    V = U.copy()
    with fvg.Solver(cfg) as s:
        s.upload(U)

        def step():
            nonlocal t, lag
            r = s.step(t, 1e9)
            dt, S, lag, ok = o.step(cfg, V, t, 1e9, 0.0, lag)
            t += dt
            assert ok and r.dt == dt and r.s_max == S and same(s.download(), V)

        step()
        for half in (1e-3, 0.0, 2e-3):
            R, S = s.residual(half)
            Ro, So = o.residual(cfg, V, half)
            assert S == So and same(R, Ro)
            if cfg.time_scheme != 3:   # a MUSCL-Hancock step would take its residual's speed
                step()
