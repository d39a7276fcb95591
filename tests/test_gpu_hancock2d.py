"""k_hancock_step2d (a MUSCL-Hancock step of a periodic 2-D mesh in one launch): meshes of one tile, smaller than a tile,
ragged on either axis and of two cells, by single steps, eager and replayed runs in either parity and past the end of a
run, each against the oracle bit for bit; and tiles with values outside the in-range arithmetic beside tiles inside."""
import numpy as np
import pytest

from cases import base_keys, shock_state, smooth_state
from fenice_amd import fvg
from oracle_lib import Oracle

pytestmark = pytest.mark.gpu


def same(a, b):
    return np.array_equal(a.view(np.uint64), b.view(np.uint64))


@pytest.mark.parametrize("over", [dict(), dict(muscl_limiter="Koren", riemann_solver="HLLC (Low-Mach Thornber)")])
@pytest.mark.parametrize("dims", [(14, 14), (2, 2), (3, 29), (15, 13), (56, 5), (43, 70)])
def test_steps(dims, over):
    keys = base_keys(*dims, time_scheme="MUSCL-Hancock", **over)
    cfg = fvg.config_from_keys(keys)
    U, o = shock_state(*dims, 1, 11), Oracle()
    V, t, lag = U.copy(), 0.0, 0.0
    with fvg.Solver(cfg) as s:
        s.upload(U)

        def follow(n, t_end=1e9):
            nonlocal t, lag
            for _ in range(n):
                dt, S, lag, ok = o.step(cfg, V, t, t_end, 0.0, lag)
                assert ok
                t += dt
            return S

        r = s.step(0.0, 1e9)
        assert r.s_max == follow(1) and r.dt == t and same(s.download(), V)
        for n in (1, 5, 8, 3):   # single steps between the runs change which plane set a graph starts from
            tt, k, S = s.advance(t, 1e9, max_steps=n)
            assert k == n and S == follow(n) and tt == t and same(s.download(), V)
            r = s.step(t, 1e9)
            assert r.s_max == follow(1) and same(s.download(), V)
        s.set_graphs(False)
        tt, k, S = s.advance(t, 1e9, max_steps=3)
        assert S == follow(3) and tt == t and same(s.download(), V)
        s.set_graphs(True)
        end = t + 2.5 * r.dt   # three steps, the graph's others and the next chunk's are past the end
        tt, k, S = s.advance(t, end)
        follow(k, end)
        assert tt == t == end and same(s.download(), V)


def test_range_is_decided_per_tile():
    n = 60
    cfg = fvg.config_from_keys(base_keys(n, n, time_scheme="MUSCL-Hancock"))
    U = smooth_state(n, n, 1, 4)
    U[(n * n) // 2:, 2] = U[(n * n) // 2:, 0] * 2.0 ** -600   # rho v of the upper half far below the range
    o, V, t, lag = Oracle(), U.copy(), 0.0, 0.0
    with fvg.Solver(cfg) as s:
        s.upload(U)
        for _ in range(4):
            r = s.step(t, 1e9)
            dt, S, lag, ok = o.step(cfg, V, t, 1e9, 0.0, lag)
            t += dt
            assert ok and r.s_max == S and same(s.download(), V)
