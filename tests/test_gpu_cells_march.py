"""k_cells_march (several planes per thread on a periodic viscous 3-D mesh) at plane counts that leave a ragged last
segment, divide evenly, or just reach the rule's threshold: FP64 residual and step against the oracle bit for bit, FP32
within the residual bound of the FP32 mode."""
import numpy as np
import pytest

from cases import base_keys, smooth_state
from fenice_amd import fvg
from oracle_lib import Oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(20, 128, 130), (33, 256, 67), (9, 512, 40), (70, 128, 64)])
def test_periodic_viscous_mesh(dims):
    keys = base_keys(*dims, reconstruction="weno5", use_viscous="true", mu="6.25e-4", pr="0.71")
    U = smooth_state(*dims, 3, mach=0.1)
    cfg = fvg.config_from_keys(keys)
    o = Oracle()
    Ro, So = o.residual(cfg, U)
    with fvg.Solver(cfg) as s:
        s.upload(U)
        R, S = s.residual()
        assert S == So and np.array_equal(R.view(np.uint64), Ro.view(np.uint64))
        s.step(0.0, 1.0)
        D = s.download()
    o.step(cfg, U1 := U.copy(), 0.0, 1.0)
    assert np.array_equal(D.view(np.uint64), U1.view(np.uint64))
    with fvg.Solver(fvg.config_from_keys(dict(keys, flux_precision="fp32"))) as s:
        s.upload(U)
        R, S = s.residual()
    assert abs(S - So) < 1e-5 * So
    assert (np.abs(R - Ro).max(0) < 2e-4 * np.abs(Ro).max(0)).all()
