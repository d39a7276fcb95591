"""MUSCL-Hancock residuals whose half step carries the advanced states out of the range of the in-range FP64 operations
(fvg_residual takes any half step): the faces fall back to the plain operations, with the oracle's values and NaNs."""
import numpy as np
import pytest

from cases import base_keys
from fenice_amd import fvg
from oracle_lib import Oracle

pytestmark = pytest.mark.gpu

WALLS = dict(bc_xmin="wall", bc_xmax="transmissive", bc_ymin="no_slip", bc_ymax="wall")


def converging(nx, ny, nz):
    """A gas at rest but for the last axis' velocity +1, 0, -1 in repetition: at the cells of 0 the momentum fluxes of
    both sides are equal, so a half step raises their density and energy without limit and leaves them admissible."""
    n = nx * ny * nz
    k = np.arange(n) // (nx if nz == 1 else nx * ny)
    v = np.array([1.0, 0.0, -1.0])[k % 3]
    U = np.zeros((n, 5))
    U[:, 0] = 1000.0
    U[:, 2 if nz == 1 else 4] = 1000.0 * v
    U[:, 3] = 2.5 + 500.0 * v * v
    return U


def agree(a, b):
    return np.array_equal(np.isnan(a), np.isnan(b)) and np.array_equal(np.where(np.isnan(a), 0.0, a), np.where(np.isnan(b), 0.0, b))


@pytest.mark.parametrize("half", [1e-3, 2.0 ** 190, 2.0 ** 201, 2.0 ** 500, 1e307])
@pytest.mark.parametrize("dims,over", [
    ((14, 12, 1), {}), ((31, 33, 1), {}), ((14, 12, 1), dict(riemann_solver="HLLC (Low-Mach Thornber)", shock_blend="0.2")),
    ((12, 9, 1), dict(periodic=False, boundary_order=2, **WALLS)), ((7, 6, 9), {}),
    ((7, 6, 9), dict(periodic=False, bc_zmin="wall", bc_zmax="no_slip", **WALLS))])
def test_residual_of_any_half_step(dims, over, half):
    cfg = fvg.config_from_keys(base_keys(*dims, time_scheme="MUSCL-Hancock", **over))
    U, o = converging(*dims), Oracle()
    with fvg.Solver(cfg) as s:
        s.upload(U)
        R, S = s.residual(half)
        Ro, So = o.residual(cfg, U, half)
        assert S == So and agree(R, Ro)
        s.upload(U)   # the fall-back is the residual's own: the next one is in range again
        R, S = s.residual(1e-3)
        Ro, So = o.residual(cfg, U, 1e-3)
        assert S == So and np.array_equal(R, Ro)


@pytest.mark.parametrize("dims", [(14, 12), (31, 33)])
def test_step_of_any_length(dims):
    """The same by a step of the periodic 2-D mesh (k_hancock_step2d), whose CFL number makes it as long."""
    cfg = fvg.config_from_keys(base_keys(*dims, time_scheme="MUSCL-Hancock", cfl="8e307"))
    U, o = converging(*dims, 1), Oracle()
    V = U.copy()
    dt, So, lag, ok = o.step(cfg, V, 0.0, 1e308, 0.0, 0.0)
    assert ok
    with fvg.Solver(cfg) as s:
        s.upload(U)
        r = s.step(0.0, 1e308)
        assert r.dt == dt and r.s_max == So and agree(s.download(), V)
