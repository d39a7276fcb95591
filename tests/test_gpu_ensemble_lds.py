"""Device tests: 1-D ensembles whose chunks fit in LDS take the same bits as ensembles in global memory."""
import numpy as np
import pytest

from fenice_amd.workloads import ensemble_keys, riemann_ensemble, riemann_states
from test_gpu_ensemble import SCHEMES, run_teams, same, say

pytestmark = pytest.mark.gpu


# ---- chunks in LDS (k_ensemble_lds): an instance too large for it takes the whole ensemble through global memory -------
@pytest.mark.parametrize("teams", [(1, 512, False), (4, 3, True), (16, 40, True)], ids=["single", "teams4", "teams16"])
@pytest.mark.parametrize("name,over", [s for s in SCHEMES if s[1].get("reconstruction") != "none"],
                         ids=[s[0] for s in SCHEMES if s[1].get("reconstruction") != "none"])
def test_lds_chunks_match_global_memory(name, over, teams):
    # sizes around the stencil, the wavefront and the workgroup, with values outside the range of the shorter
    # operations (a velocity of 1e-125, an energy of 1e32) in two of them; the same arithmetic, so the same bits
    say("ensemble LDS against global memory", name, teams)
    keys = dict(ensemble_keys(), **over)
    _, _, params = riemann_ensemble(12, seed=31, nmin=2, nmax=3)
    n = np.array([1, 2, 3, 6, 7, 63, 64, 65, 190, 257, 700, 3500], dtype=np.int32)   # 3,500 cells: 168 KB
    U = riemann_states(n, params)
    off = np.concatenate([[0], np.cumsum(n)])
    U[off[5] + 20:off[5] + 40, 1] = 1e-125
    U[off[7] + 30, 3] = 1e32
    outs = []
    for k in (11, 12):
        Ud, r, _, _ = run_teams(keys, n[:k], U[:off[k]], 0.05, 40, teams, 256)
        outs.append((Ud[:off[11]], r.t[:11], r.steps[:11], r.s_last[:11], r.diverged[:11]))
    for a, b in zip(*outs):
        assert same(np.asarray(a, dtype=np.float64), np.asarray(b, dtype=np.float64))


def test_largest_lds_chunk_matches_global_memory():
    say("ensemble: largest chunk in LDS")
    _, _, params = riemann_ensemble(2, seed=33, nmin=2, nmax=3)
    n = np.array([3400, 3500], dtype=np.int32)
    U = riemann_states(n, params)
    for teams in ((1, 512, False), (3, 100, True)):
        a, ra, _, _ = run_teams(ensemble_keys(), n[:1], U[:3400], 0.05, 30, teams, 1024)
        b, rb, _, _ = run_teams(ensemble_keys(), n, U, 0.05, 30, teams, 1024)
        assert same(a, b[:3400]) and ra.t[0] == rb.t[0] and ra.s_last[0] == rb.s_last[0]
