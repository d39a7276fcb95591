"""Which kernel and how much LDS a 1-D ensemble takes: the whole instance where workgroups are limited by their registers
anyway, the chunks of teams where one long instance would take the LDS of many short ones, global memory where that is
shorter or an instance is too large; each with the same bits."""
import numpy as np
import pytest

from fenice_amd import fvg
from fenice_amd.workloads import ensemble_keys, riemann_ensemble, riemann_states
from test_gpu_ensemble import SCHEMES, same, say

pytestmark = pytest.mark.gpu


def states(n, seed=5):
    _, _, params = riemann_ensemble(len(n), seed=seed, nmin=2, nmax=3)
    return np.array(n, dtype=np.int32), riemann_states(np.array(n, dtype=np.int32), params)


def launch(n, U, block, steps, teams=None, over={}):
    with fvg.Ensemble(fvg.config_from_keys(dict(ensemble_keys(), **over)), n) as e:
        e.block = block
        if teams:
            e.set_teams(*teams)
        e.upload(U)
        r = e.run(1e9, steps)
        return e.download(3), r, e.lds_cells, e.plan


@pytest.mark.parametrize("block,room", [(64, 300), (128, 600), (256, 1100), (512, 3000)])
def test_one_long_instance_among_short_ones(block, room):
    say("ensemble choice: one of 3,000 among 4,000 of 128 cells", block)
    n, U = states([3000] + [128] * 4000)
    Ud, r, cells, plan = launch(n, U, block, 4)
    if block < 512:   # 3, 6 and 12 workgroups fit a CU
        assert plan[0] == 1 and 128 <= cells <= room
    else:
        assert cells == 3000
    m, V = np.append(n, 3500).astype(np.int32), np.concatenate([U, states([3500], 6)[1]])
    Vd, q, cells, _ = launch(m, V, block, 4)   # global memory
    assert cells == 0 and same(Ud, Vd[:len(Ud)]) and same(r.t, q.t[:-1]) and same(r.s_last, q.s_last[:-1])


def test_long_instances_in_short_workgroups():
    say("ensemble choice: 600 of 3,000 cells")
    n, U = states([3000] * 600)
    a, ra, cells, _ = launch(n, U, 64, 3)
    assert cells == 0   # no team is left to split them, and one wavefront a CU is slower than eight
    b, rb, cells, _ = launch(n, U, 768, 3)
    assert cells == 3000 and same(a, b) and same(ra.t, rb.t)


@pytest.mark.parametrize("teams", [None, (1, 512)])
def test_equal_instances_stay_in_lds(teams):
    n, U = states([128] * 500)
    for block in (64, 256, 1024):
        assert launch(n, U, block, 2, teams)[2] == 128


def test_sizes_of_the_lds_tests():
    """The ensembles that test_gpu_ensemble_lds compares are one in LDS and one in global memory."""
    n, U = states([1, 2, 3, 6, 7, 63, 64, 65, 190, 257, 700, 3500])
    for name, over in SCHEMES:
        if over.get("reconstruction") == "none":
            continue
        for teams in ((1, 512, False), (4, 3, True), (16, 40, True)):
            k = len(U) - 3500
            assert launch(n[:11], U[:k], 256, 2, teams, over)[2] > 0, (name, teams)
            assert launch(n, U, 256, 2, teams, over)[2] == 0, (name, teams)
    n, U = states([3400, 3500])
    for teams in ((1, 512, False), (3, 100, True)):
        assert launch(n[:1], U[:3400], 1024, 2, teams)[2] == 3400
        assert launch(n, U, 1024, 2, teams)[2] == 0


def test_tuned_block_is_kept_for_the_same_kernel_and_teams(tmp_path):
    say("ensemble choice: tuner's cache")
    n, U = states([64] * 40)
    cache = tmp_path / "tune.txt"

    def tune(teams=None):
        with fvg.Ensemble(fvg.config_from_keys(ensemble_keys()), n) as e:
            if teams:
                e.set_teams(*teams)
            e.upload(U)
            return e.tune(0.002, 20, str(cache))[1]

    assert not tune() and tune()
    assert not tune(teams=(1, 512)) and tune(teams=(1, 512)) and not tune(teams=(4, 20)) and not tune(teams=(4, 20, True))
    key, rest = cache.read_text().splitlines()[0].split(" ", 1)
    cache.write_text(key[:key.index("|lds")] + " " + rest + "\n")   # a line that does not say which kernel it was for
    assert not tune()
