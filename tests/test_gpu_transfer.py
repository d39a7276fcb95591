"""Uploads and downloads (fvg_transfer.hip): every bit of a state comes back, at sizes around the staging's chunks and
lanes (below one chunk, several chunks of one lane, several lanes with a ragged end) and for every component count."""
import numpy as np
import pytest

from cases import base_keys
from fenice_amd import fvg
from fenice_amd.workloads import ensemble_keys

pytestmark = pytest.mark.gpu


def bits(n, nq, seed):
    """Random bit patterns (subnormals, infinities and NaN among them)."""
    return np.random.default_rng(seed).integers(0, 1 << 64, size=(n, nq), dtype=np.uint64).view(np.float64)


def same(a, b):
    return np.array_equal(np.ascontiguousarray(a).view(np.uint64), np.ascontiguousarray(b).view(np.uint64))


@pytest.mark.parametrize("dims", [(7, 3, 1), (5, 3, 3), (181, 182, 1), (239, 137, 1), (101, 75, 52), (1451, 1021, 1)])
def test_state_round_trip(dims):
    n = dims[0] * dims[1] * dims[2]
    with fvg.Solver(fvg.config_from_keys(base_keys(*dims))) as s:
        for seed, nq in enumerate((5,) if dims[2] > 1 else (4, 5)):
            U = bits(n, nq, seed)
            s.upload(U)
            D = s.download(5)
            k = 5 if dims[2] > 1 else 4
            assert same(D[:, :k], U[:, :k])
            if k == 4:
                assert same(D[:, 4], np.zeros(n)) and same(s.download(4), U[:, :4])


@pytest.mark.parametrize("sizes", [[3, 5, 4], [4099, 8191, 128], [70001, 500003, 9]])
def test_ensemble_round_trip(sizes):
    n = sum(sizes)
    with fvg.Ensemble(fvg.config_from_keys(ensemble_keys()), sizes) as e:
        for nq in (3, 4, 5):
            U = bits(n, nq, nq)
            e.upload(U)
            keep = [0, 1, 2] if nq == 3 else [0, 1, 3]
            assert same(e.download(3), U[:, keep])
            D = e.download(5)
            assert same(D[:, [0, 1, 3]], U[:, keep]) and same(D[:, [2, 4]], np.zeros((n, 2)))
