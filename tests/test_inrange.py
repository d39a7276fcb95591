"""The in-range FP64 operations of the face kernels (fvg_device.hpp): divisions by a constant against the IEEE division
on the host, and on the device the residual of fields at both edges of value_in_range against the oracle."""
import os
import shutil
import subprocess

import numpy as np
import pytest

from cases import base_keys
from oracle_lib import Oracle

HERE = os.path.dirname(os.path.abspath(__file__))
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


def test_by_const_equals_the_ieee_division(tmp_path):
    if not os.path.exists(HIPCC):
        pytest.skip("hipcc not found")
    exe = str(tmp_path / "inrange_check")
    subprocess.run([HIPCC, "-x", "hip", "-O2", "-std=c++17", "-ffp-contract=off", "--offload-arch=gfx950",
                    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
                    os.path.join(HERE, "inrange_check.cpp"), "-o", exe], check=True, capture_output=True)
    r = subprocess.run([exe, "400000", "3"], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and "differing: 0, bounds ok" in r.stdout, r.stdout


def edge_state(nx, ny, nz, edge, seed=5):
    """A smooth field whose velocities are tiny multiples of an edge of value_in_range, or whose density and pressure
    lie at its upper edge."""
    rng = np.random.default_rng(seed)
    n = nx * ny * nz
    rho, p = 1.0 + 0.3 * rng.random(n), 1.0 + 0.3 * rng.random(n)
    u, v, w = (rng.standard_normal(n) for _ in range(3))
    if edge in ("low-in", "low-out"):   # |v| in [1, 2) 2^-400 (in range) or 2^-401 (out)
        s = 2.0 ** (-400 if edge == "low-in" else -401)
        v = np.sign(v) * (1.0 + rng.random(n)) * s
        w = np.where(rng.random(n) < 0.5, 0.0, v)
    elif edge in ("high-in", "high-out"):   # p in [1, 2) 2^99 or 2^100 with rho of order one: speeds of 2^50
        p = (1.0 + 0.99 * rng.random(n)) * 2.0 ** (99 if edge == "high-in" else 100)
        u, v, w = (x * 2.0 ** 45 for x in (u, v, w))
    else:   # zeros of both signs among the velocities
        v = np.where(rng.random(n) < 0.5, -0.0, 0.0)
        w = np.where(rng.random(n) < 0.7, -0.0, rng.standard_normal(n))
    U = np.empty((n, 5))
    U[:, 0], U[:, 1], U[:, 2], U[:, 4] = rho, rho * u, rho * v, (rho * w if nz > 1 else 0.0)
    U[:, 3] = p / 0.4 + 0.5 * rho * (u * u + v * v + (w * w if nz > 1 else 0.0))
    return U


@pytest.mark.gpu
@pytest.mark.parametrize("edge", ["low-in", "low-out", "high-in", "high-out", "zeros"])
@pytest.mark.parametrize("dims,over", [
    ((13, 9, 1), dict(reconstruction="weno5")), ((9, 8, 7), dict(reconstruction="weno5", use_viscous="true", mu="0.01")),
    ((13, 9, 1), dict(reconstruction="muscl", muscl_limiter="Koren")), ((9, 8, 7), dict(reconstruction="muscl")),
    ((9, 8, 7), dict(reconstruction="weno3", riemann_solver="HLLC (Low-Mach Thornber)")),
    ((9, 8, 7), dict(reconstruction="weno5", flux_quadrature="fourth")),
    ((14, 12, 1), dict(time_scheme="MUSCL-Hancock")),
])
def test_residual_at_the_edges_of_the_range(edge, dims, over):
    from fenice_amd import fvg
    cfg = fvg.config_from_keys(base_keys(*dims, **over))
    U = edge_state(*dims, edge)
    o = Oracle()
    half = 1e-3 if cfg.time_scheme == 3 else 0.0
    if half and edge.startswith("high"):
        half *= 2.0 ** -50
    with fvg.Solver(cfg) as s:
        s.upload(U)
        R, S = s.residual(half)
        Ro, So = o.residual(cfg, U, half)
    assert S == So
    assert np.array_equal(R.view(np.uint64), Ro.view(np.uint64))
