"""The mean density of a mass-flow side (k_sides) over sides around one and several of its chunks of 2,048 cells, from each
direction: the residual has the oracle's bits, which the inflow velocity of every boundary face enters."""
import numpy as np
import pytest

from cases import base_keys, smooth_state
from fenice_amd import fvg
from oracle_lib import Oracle

pytestmark = pytest.mark.gpu

IO = dict(u_in="0.3", v_in="0.1", rho_in="1.2", p_out="0.9", bc_zmin="periodic", bc_zmax="periodic")
X = dict(IO, bc_xmin="massflow_inlet", bc_xmax="nonreflecting", bc_ymin="wall", bc_ymax="no_slip")
XR = dict(IO, bc_xmax="massflow_inlet", bc_xmin="transmissive", bc_ymin="wall", bc_ymax="no_slip")
Y = dict(IO, bc_ymin="massflow_inlet", bc_ymax="nonreflecting", bc_xmin="wall", bc_xmax="no_slip")
YR = dict(IO, bc_ymax="massflow_inlet", bc_ymin="massflow_inlet", bc_xmin="wall", bc_xmax="no_slip")


@pytest.mark.parametrize("dims,sides", [((4, n, 1), X) for n in (1, 63, 2047, 2048, 2049, 4096, 6177)] + [
    ((4, 2111, 1), XR), ((4097, 3, 1), Y), ((2080, 3, 1), YR), ((3, 70, 65), X), ((61, 3, 70), YR)])
def test_side_mean(dims, sides):
    cfg = fvg.config_from_keys(base_keys(*dims, periodic=False, **sides))
    U = smooth_state(*dims, 9)
    Ro, So = Oracle().residual(cfg, U)
    with fvg.Solver(cfg) as s:
        s.upload(U)
        R, S = s.residual()
    assert S == So and np.array_equal(R.view(np.uint64), Ro.view(np.uint64))
