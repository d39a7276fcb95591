"""The work that a user of this framework has it do, as cases to be timed: runs on a uniform mesh (`Solver`) and
ensembles of independent runs (`Ensemble`), through the public entry points of `fenice_amd.fvg`.

A pass is a whole call on host data, as the C ABI takes it: the state goes up, the run advances, the state comes back
(`upload`, `advance` or `step` or `residual`, `download`). The state crosses the boundary as the array of cells that the
reference holds, so both conversions and both copies are part of what a user waits for. A program keeps its context
(`Solver`, `Ensemble`), the network's weights and the tuned workgroup size; `prepare` makes those.

Every run of a family starts from the family's flow with seeded phases and a seeded disturbance, so another seed is
another flow of the same kind.

`exact` restates the schemes in plain torch at 64 bits: every face of an axis at once, boundary conditions as padded
arrays. It shares no code with the package, and follows the published formulas (WENO-Z, HLLC with Einfeldt bounds,
SSP Runge-Kutta, MUSCL-Hancock), not the device's layout.
"""
from __future__ import annotations

import math
import os

import numpy as np
import torch

from fenice_amd import fvg, workloads

TWO_PI = 2.0 * math.pi
FAR = 1e9   # an end time that the step limit reaches first


# ----------------------------------------------------------------------------------------------------------------
# The cases
# ----------------------------------------------------------------------------------------------------------------
def listed():
    return [
        # the lid-driven cavity stepped one call at a time, as the reference's own loop would through its time-scheme
        # interface: small meshes, a host round trip per step, launches and latency
        dict(name="cavity_64_step", family="cavity", nx=64, ny=64, recon="muscl", steps=20),
        # the isentropic vortex under MUSCL-Hancock: an ordinary 2-D run of many cheap steps
        dict(name="vortex_256_hancock", family="vortex", nx=256, ny=256, steps=160),
        # one residual of a 3-D mesh of odd sizes with walls and ghost slabs, as a caller with its own time integrator
        # asks for it
        dict(name="residual_101x75x52", family="residual", nx=101, ny=75, nz=52, recon="weno3", lowmach=True),
        # a duct with a mass-flow inlet, a non-reflecting outlet and no-slip walls: the boundary conditions of an
        # internal flow, viscous, WENO5-Z
        dict(name="duct_160x64x48", family="duct", nx=160, ny=64, nz=48, steps=20),
        # the Kelvin-Helmholtz layer at its benchmark size: a large inviscid 2-D run
        dict(name="kh_2048_fp64", family="kh", nx=2048, ny=2048, flux="fp64", steps=40),
        # the 3-D Taylor-Green vortex at its benchmark size and precision, with a monitor row at the end (the largest)
        dict(name="tgv_256_fp64", family="tgv", nx=256, ny=256, nz=256, flux="fp64", learned=False, quad="midpoint", steps=20,
             monitor=True),
        # the same flow with FP32 fluxes at 192^3
        dict(name="tgv_192_fp32", family="tgv", nx=192, ny=192, nz=192, flux="fp32", learned=False, quad="midpoint", steps=50,
             monitor=False),
        # the learned troubled-face indicator, FP64 and FP32 fluxes, the second on a box of uneven, odd sizes
        dict(name="tgv_128_fp64_learned", family="tgv", nx=128, ny=128, nz=128, flux="fp64", learned=True, quad="midpoint",
             steps=60, monitor=False),
        dict(name="tgv_145x130x171_fp32_learned", family="tgv", nx=145, ny=130, nz=171, flux="fp32", learned=True,
             quad="midpoint", steps=60, monitor=False),
        # the fourth-order flux quadrature
        dict(name="tgv_96_fourth", family="tgv", nx=96, ny=96, nz=96, flux="fp64", learned=False, quad="fourth", steps=40,
             monitor=False),
        # ensembles of 1-D Riemann problems and of 2-D vortices of uneven sizes, each run to its end time
        dict(name="riemann_512x128..2048", family="riemann", ninst=512, nmin=128, nmax=2048, t_end=0.02),
        dict(name="vortices_96x32..192", family="vortices", ninst=96, nmin=32, nmax=192, t_end=0.3),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _box(rng, lo, hi):
    """Three sizes around a common one, odd ones among them."""
    n = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return [max(12, min(256, int(round(n * rng.uniform(0.75, 1.33))))) for _ in range(3)]


def _steps(cells, budget, most):
    return max(4, min(most, int(budget / cells)))


def draw(rng):
    f = rng.choice(["cavity", "vortex", "residual", "duct", "kh", "kh", "tgv", "tgv", "tgv", "tgv", "riemann", "vortices"])
    if f == "cavity":
        return dict(family=f, nx=_log_int(rng, 20, 200), ny=_log_int(rng, 20, 200), recon=rng.choice(["muscl", "weno3", "weno5"]),
                    steps=rng.randint(8, 30))
    if f == "vortex":
        nx, ny = _log_int(rng, 48, 1024), _log_int(rng, 48, 1024)
        return dict(family=f, nx=nx, ny=ny, steps=_steps(nx * ny, 2e7, 160))
    if f == "residual":
        nx, ny, nz = _box(rng, 20, 160)
        return dict(family=f, nx=nx, ny=ny, nz=nz, recon=rng.choice(["muscl", "weno3", "weno5"]), lowmach=rng.random() < 0.5)
    if f == "duct":
        nx, ny, nz = 2 * _log_int(rng, 24, 110), _log_int(rng, 20, 100), _log_int(rng, 20, 100)
        return dict(family=f, nx=nx, ny=ny, nz=nz, steps=_steps(nx * ny * nz, 1e7, 20))
    if f == "kh":
        nx, ny = _log_int(rng, 96, 2048), _log_int(rng, 96, 2048)
        return dict(family=f, nx=nx, ny=ny, flux=rng.choice(["fp64", "fp64", "fp32"]), steps=_steps(nx * ny, 1.6e8, 80))
    if f == "tgv":
        kind = rng.choice(["fp64", "fp64", "fp32", "learned64", "learned32", "fourth"])
        nx, ny, nz = _box(rng, 64 if kind.startswith("learned") else 24, 110 if kind == "fourth" else 190)
        return dict(family=f, nx=nx, ny=ny, nz=nz, flux="fp32" if kind in ("fp32", "learned32") else "fp64",
                    learned=kind.startswith("learned"), quad="fourth" if kind == "fourth" else "midpoint",
                    steps=_steps(nx * ny * nz, 4e7 if kind == "fourth" else 1.2e8, 60), monitor=kind == "fp64" and rng.random() < 0.5)
    if f == "riemann":
        nmax = _log_int(rng, 300, 3000)
        return dict(family=f, ninst=_log_int(rng, 64, 900), nmin=min(128, nmax // 2), nmax=nmax, t_end=0.02 * min(1.0, 1500.0 / nmax))
    nmax = _log_int(rng, 40, 224)
    return dict(family="vortices", ninst=_log_int(rng, 16, 160), nmin=max(8, nmax // 6), nmax=nmax, t_end=0.3)


# ----------------------------------------------------------------------------------------------------------------
# The run keys (the reference's names and labels) and the initial flows
# ----------------------------------------------------------------------------------------------------------------
def _keys(c):
    f = c["family"]
    if f == "cavity":   # air-like gas at rest under a moving lid, Mach about 0.08
        return dict(nx=c["nx"], ny=c["ny"], nz=1, Lx=1.0, Ly=1.0, gamma=1.4, use_viscous="true", mu=2.5e-3, pr=0.72, bc_xmin="no_slip",
                    bc_xmax="no_slip", bc_ymin="no_slip", bc_ymax="moving_wall", u_in=1.0, rho_in=1.0, p_out=100.0,
                    riemann_solver="HLLC (Low-Mach Thornber)", reconstruction=c["recon"], muscl_limiter="Van Leer",
                    time_scheme="SSP Runge-Kutta 3", cfl=0.4, boundary_order=2)
    if f == "vortex":
        return dict(workloads.vortex_keys(c["nx"], cfl="0.7"), ny=c["ny"])
    if f == "residual":
        return dict(nx=c["nx"], ny=c["ny"], nz=c["nz"], Lx=TWO_PI, Ly=TWO_PI, Lz=TWO_PI, gamma=1.4, use_viscous="true", mu=0.01, pr=0.71,
                    bc_xmin="transmissive", bc_xmax="wall", bc_ymin="no_slip", bc_ymax="wall", bc_zmin="periodic", bc_zmax="periodic",
                    riemann_solver="HLLC (Low-Mach Thornber)" if c["lowmach"] else "HLLC", reconstruction=c["recon"],
                    muscl_limiter="Van Leer", time_scheme="SSP Runge-Kutta 3", cfl=0.5, boundary_order=2)
    if f == "duct":
        return dict(nx=c["nx"], ny=c["ny"], nz=c["nz"], Lx=4.0, Ly=1.0, Lz=1.0, gamma=1.4, use_viscous="true", mu=1e-3, pr=0.72,
                    bc_xmin="massflow_inlet", bc_xmax="nonreflecting", bc_ymin="no_slip", bc_ymax="no_slip", bc_zmin="periodic",
                    bc_zmax="periodic", u_in=0.3, v_in=0.0, rho_in=1.0, p_out=1.0, riemann_solver="HLLC", reconstruction="weno5",
                    time_scheme="SSP Runge-Kutta 3", cfl=0.5, boundary_order=2)
    if f == "kh":
        k = dict(workloads.kh_keys(c["nx"]), ny=c["ny"])
        if c["flux"] != "fp64":
            k["flux_precision"] = c["flux"]
        return k
    if f == "tgv":
        k = dict(workloads.taylor_green_keys(c["nx"], flux=c["flux"], quadrature=c["quad"]), ny=c["ny"], nz=c["nz"])
        if c["learned"]:
            k["indicator"] = "learned"
        return k
    if f == "riemann":
        return workloads.ensemble_keys(t_end=c["t_end"])
    return workloads.vortex_ensemble_keys(**{a: str(c[a]) for a in ("nx", "ny") if a in c})


def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _axes(nx, ny, nz):
    d = _device()
    ax = [(torch.arange(n, dtype=torch.float64, device=d) + 0.5) / n for n in (nx, ny, nz)]
    return ax[0].view(1, 1, -1), ax[1].view(1, -1, 1), ax[2].view(-1, 1, 1)


def _rng(seed):
    g = torch.Generator()
    g.manual_seed(int(seed) * 7919 + 17)
    return lambda *shape: torch.rand(*shape, generator=g, dtype=torch.float64)


def _disturbance(r, x, y, z, modes=4):
    """A sum of a few long seeded waves of unit size in the box."""
    out = 0.0
    for _ in range(modes):
        k = [int(v) for v in (r(3) * 3).floor() + 1]
        a, b, c = (float(v) * TWO_PI for v in r(3))
        out = out + torch.sin(TWO_PI * k[0] * x + a) * torch.cos(TWO_PI * k[1] * y + b) * torch.cos(TWO_PI * k[2] * z + c)
    return out / modes


def _cells(rho, u, v, w, p, gamma, ncomp):
    """The array of cells (n, ncomp) on the host."""
    rho, u, v, w, p = torch.broadcast_tensors(rho, u, v, w, p)
    comps = [rho, rho * u, rho * v, p / (gamma - 1.0) + 0.5 * rho * (u * u + v * v + w * w), rho * w][:ncomp]
    return torch.stack([t.reshape(-1) for t in comps], dim=1).cpu().numpy()


def _sizes(c):
    """Cells (a side) of an ensemble's instances: the case's own, whatever the flow's seed."""
    u = workloads.unit_doubles(c["ninst"], c["ninst"])
    return (c["nmin"] + np.floor(u * (c["nmax"] - c["nmin"] + 1))).astype(np.int32)


def _vortex(nx, ny, cx, cy, L=10.0):
    """The isentropic vortex, beta 5 in the free stream (1, 1) on [0, L]^2, centred at (cx, cy) L."""
    i, j = np.arange(nx)[None, :], np.arange(ny)[:, None]
    dx, dy = (i + 0.5) / nx - cx, (j + 0.5) / ny - cy
    dx, dy = L * (dx - np.round(dx)), L * (dy - np.round(dy))
    r2 = dx * dx + dy * dy
    g = 5.0 / TWO_PI * np.exp(0.5 * (1.0 - r2))
    T = 1.0 - 0.4 * 25.0 / (8.0 * 1.4 * math.pi ** 2) * np.exp(1.0 - r2)
    rho, u, v = T ** 2.5, 1.0 - g * dy, 1.0 + g * dx
    return np.stack([t.ravel() for t in (rho, rho * u, rho * v, rho * T / 0.4 + 0.5 * rho * (u * u + v * v))], axis=1)


def _flow(c, seed):
    f, r = c["family"], _rng(seed)
    if f == "riemann":
        n = _sizes(c)
        params = workloads.riemann_ensemble(c["ninst"], seed=int(seed) + 1, nmin=2, nmax=3)[2]
        return n, workloads.riemann_states(n, params)
    if f == "vortices":
        n = _sizes(c)
        return n, np.concatenate([_vortex(int(k), int(k), float(a), float(b)) for k, (a, b) in zip(n, r(len(n), 2))])
    nz = c.get("nz", 1)
    x, y, z = _axes(c["nx"], c["ny"], nz)
    zero, one = torch.zeros_like(x), torch.ones_like(x)
    if f == "cavity":
        a = float(r(1)) * TWO_PI
        u = 0.3 * torch.sin(math.pi * x) * torch.sin(TWO_PI * y + a)
        v = 0.3 * torch.sin(TWO_PI * x + a) * torch.sin(math.pi * y)
        return _cells(1.0 + 0.01 * _disturbance(r, x, y, zero), u, v, zero, 100.0 + 0.1 * _disturbance(r, x, y, zero), 1.4, 4)
    if f == "vortex":
        return _vortex(c["nx"], c["ny"], float(r(1)), float(r(1)))
    if f == "residual":   # subsonic waves with a moderate jump across a seeded plane
        s = 0.3 + 0.4 * float(r(1))
        jump = torch.where(x + 0.2 * torch.sin(TWO_PI * y) < s, 1.0, 0.6)
        d = [_disturbance(r, x, y, z) for _ in range(5)]
        return _cells(jump + 0.1 * d[0], 0.3 * d[1], 0.3 * d[2], 0.3 * d[3], jump * (1.0 + 0.1 * d[4]), 1.4, 5)
    if f == "duct":   # a flat profile between the walls with seeded waves
        prof = 0.3 * (1.0 - (2.0 * y - 1.0) ** 8)
        d = [_disturbance(r, x, y, z) for _ in range(4)]
        return _cells(one + 0.01 * d[0], prof * (1.0 + 0.2 * d[1]), 0.02 * d[2], 0.02 * d[3], one + 0.01 * d[0], 1.4, 5)
    if f == "kh":
        inner = ((y - 0.5).abs() < 0.25).expand(1, c["ny"], c["nx"])
        noise = 1e-3 * (2.0 * r(1, c["ny"], c["nx"]).to(x.device) - 1.0)
        a = float(r(1)) * TWO_PI
        return _cells(torch.where(inner, 2.0 * one, one), torch.where(inner, -0.5 * one, 0.5 * one),
                      0.01 * torch.sin(2.0 * TWO_PI * x + a) + noise, zero, 2.5 * one, 1.4, 4)
    a, b, g = (float(v) * TWO_PI for v in r(3))   # Taylor-Green at Mach 0.1, shifted, with 1 % of long waves
    X, Y, Z = TWO_PI * x + a, TWO_PI * y + b, TWO_PI * z + g
    d = [0.01 * _disturbance(r, x, y, z) for _ in range(3)]
    u = torch.sin(X) * torch.cos(Y) * torch.cos(Z) + d[0]
    v = -torch.cos(X) * torch.sin(Y) * torch.cos(Z) + d[1]
    p = 1.0 / (1.4 * 0.01) + (torch.cos(2 * X) + torch.cos(2 * Y)) * (torch.cos(2 * Z) + 2.0) / 16.0
    return _cells(one, u, v, d[2], p, 1.4, 5)


# ----------------------------------------------------------------------------------------------------------------
# prepare and run
# ----------------------------------------------------------------------------------------------------------------
def _weights():
    d = np.load(os.path.join(os.path.dirname(os.path.abspath(fvg.__file__)), "indicator_weights.npz"), allow_pickle=False)
    return d["params"], float(d["threshold"])


def prepare(case, seed):
    f = case["family"]
    cfg = fvg.config_from_keys(_keys(case))
    if f in ("riemann", "vortices"):
        n, U = _flow(case, seed)
        e = fvg.Ensemble(cfg, n) if f == "riemann" else fvg.Ensemble(cfg, n, ny=n)
        e.upload(U)
        e.tune(0.05 * case["t_end"], 1 << 20)
        return dict(case=case, e=e, U=U)
    s = fvg.Solver(cfg)
    weights = None
    if case.get("learned"):
        weights = _weights()
        s.set_indicator(*weights)
    return dict(case=case, s=s, U=_flow(case, seed), weights=weights)


def run(state):
    c, U = state["case"], state["U"]
    f = c["family"]
    if f in ("riemann", "vortices"):
        e = state["e"]
        e.upload(U)
        r = e.run(c["t_end"], 1 << 20)
        return dict(U=e.download(3 if f == "riemann" else 4), t=r.t, steps=r.steps, s=r.s_last)
    s = state["s"]
    s.upload(U)
    nq = U.shape[1]
    if f == "residual":
        R, smax = s.residual(ncomp=nq)
        return dict(R=R, s=smax)
    if f == "cavity":
        t, smax = 0.0, 0.0
        for _ in range(c["steps"]):
            r = s.step(t, FAR)
            t, smax = t + r.dt, r.s_max
        return dict(U=s.download(nq), t=t, s=smax)
    if f == "vortex":
        s.lagged_speed = 0.0   # a new run: the first step seeds the wave speed
    if state["weights"] is not None:
        s.set_indicator(*state["weights"])   # a new run: the audit starts over
    t, _, smax = s.advance(0.0, FAR, max_steps=c["steps"])
    out = dict(U=s.download(nq), t=t, s=smax)
    if c.get("monitor"):
        out["monitor"] = s.monitor()
    return out


def work(case):
    """One pass without what it could do without: the state up and down once, per stage of each step the compulsory state
    traffic (stage input, step start on later stages, output) and the arithmetic of the scheme, counted from its formulas
    (adds, multiplies, divisions and roots one operation each)."""
    f = case["family"]
    if f == "riemann":
        n = (case["nmin"] + case["nmax"]) / 2
        cells, nv, nd = case["ninst"] * n, 3, 1
        # steps: t_end over cfl dx / S with the family's mean largest speed (about 30)
        stages, recon = 2 * case["t_end"] * 30.0 * n / 0.5, "muscl"
    elif f == "vortices":
        n = (case["nmin"] + case["nmax"]) / 2
        cells, nv, nd = case["ninst"] * n * n, 4, 2
        stages, recon = 2 * case["t_end"] * 2.6 * n / 10.0 / 0.5, "muscl"
    else:
        nd = 2 if case.get("nz", 1) == 1 else 3
        nv = nd + 2
        cells = case["nx"] * case["ny"] * case.get("nz", 1)
        per = {"vortex": 1, "residual": 1}.get(f, 3)
        stages = per * case.get("steps", 1)
        recon = case.get("recon", "muscl" if f == "vortex" else "weno5")
    per_value = {"muscl": 12, "weno3": 30, "weno5": 95}[recon]
    face = 2 * nv * per_value + 110 + (40 if f in ("tgv", "cavity", "duct", "residual") else 0)
    cell = 20 + 8 * nv * nd + (60 if f in ("tgv", "cavity", "duct", "residual") else 0)
    if case.get("quad") == "fourth":
        face += 110 + 12 * nv * nd
    state = 8.0 * nv * cells
    rw = {"vortex": 2.0, "residual": 2.0}.get(f, 2.5 if f in ("riemann", "vortices") else 8.0 / 3.0)
    return dict(bytes=2 * state + stages * rw * state, flops=stages * cells * (nd * face + cell))


# ----------------------------------------------------------------------------------------------------------------
# exact: the schemes in plain torch at 64 bits. A state is a list [rho, rho u, rho v, rho E, rho w] of (nz, ny, nx)
# tensors; axis 0, 1, 2 is x, y, z, i.e. tensor dimension 2 - axis.
# ----------------------------------------------------------------------------------------------------------------
MOM = (1, 2, 4)


def _dim(a):
    return 2 - a


def _cut(t, a, lo, n):
    return t.narrow(_dim(a), lo, n)


class _Gas:
    def __init__(self, gamma):
        self.g = gamma

    def prim(self, U):
        rho = U[0].clamp_min(1e-10)
        u, v, w = U[1] / rho, U[2] / rho, U[4] / rho
        p = (self.g - 1.0) * (U[3] - 0.5 * rho * (u * u + v * v + w * w))
        return [rho, u, v, p.clamp_min(1e-10), w]

    def cons(self, W):
        rho, u, v, p, w = W
        return [rho, rho * u, rho * v, p / (self.g - 1.0) + 0.5 * rho * (u * u + v * v + w * w), rho * w]

    def sound(self, W):
        return torch.sqrt(self.g * W[3] / W[0])


def _safe(x):
    return torch.copysign(x.abs().clamp_min(1e-14), x)


def _hllc(gas, UL, UR, a, lowmach, blend=0.2):
    """Flux of the faces normal to axis a and their largest wave speed."""
    WL, WR = gas.prim(UL), gas.prim(UR)
    cL, cR = gas.sound(WL), gas.sound(WR)
    eL, eR = UL[3] / WL[0], UR[3] / WR[0]
    if lowmach:
        mL = torch.sqrt(WL[1] ** 2 + WL[2] ** 2 + WL[4] ** 2) / (cL + 1e-12)
        mR = torch.sqrt(WR[1] ** 2 + WR[2] ** 2 + WR[4] ** 2) / (cR + 1e-12)
        z = torch.maximum(mL, mR).clamp(1e-4, 1.0)
        for m in MOM:
            avg, half = 0.5 * (WL[m] + WR[m]), 0.5 * (WL[m] - WR[m])
            WL[m], WR[m] = avg + z * half, avg - z * half
        UL, UR = gas.cons(WL), gas.cons(WR)
        eL, eR = UL[3] / WL[0], UR[3] / WR[0]
    n = MOM[a]
    rL, rR, pL, pR, vL, vR = WL[0], WR[0], WL[3], WR[3], WL[n], WR[n]

    def flux(W, E, vn):
        F = [W[0] * vn, W[0] * W[1] * vn, W[0] * W[2] * vn, vn * (W[0] * E + W[3]), W[0] * W[4] * vn]
        F[n] = F[n] + W[3]
        return F

    FL, FR = flux(WL, eL, vL), flux(WR, eR, vR)
    SL, SR = torch.minimum(vL - cL, vR - cR), torch.maximum(vL + cL, vR + cR)
    SM = (rR * vR * (SR - vR) - rL * vL * (SL - vL) + pL - pR) / _safe(rR * (SR - vR) - rL * (SL - vL))

    def star(W, E, S, vn, p):
        k = W[0] * (S - vn) / _safe(S - SM)
        V = [k, k * W[1], k * W[2], k * (E + (SM - vn) * (SM + p / (W[0] * _safe(S - vn)))), k * W[4]]
        V[n] = k * SM
        return V

    sL, sR = star(WL, eL, SL, vL, pL), star(WR, eR, SR, vR, pR)
    F = []
    for q in range(5):
        left = torch.where(SL >= 0, FL[q], FL[q] + SL * (sL[q] - UL[q]))
        right = torch.where(SR < 0, FR[q], FR[q] + SR * (sR[q] - UR[q]))
        F.append(torch.where(SM >= 0, left, torch.where(SL >= 0, FL[q], right)))
    s = (pR - pL).abs() / torch.minimum(pL, pR)
    if bool((s > blend).any()):
        phi = torch.where(s > blend, ((s - blend) / blend).clamp_max(1.0), torch.zeros_like(s))
        for q in range(5):
            h = (SR * FL[q] - SL * FR[q] + SL * SR * (UR[q] - UL[q])) / (SR - SL)
            h = torch.where(SL >= 0, FL[q], torch.where(SR <= 0, FR[q], h))
            F[q] = (1.0 - phi) * F[q] + phi * h
    return F, float(torch.maximum(SL.abs(), SR.abs()).max())


def _weno5_weights(c, eps_rel, mean=None):
    c0, c1, c2, c3, c4 = c
    m = (c0 * c0 + c1 * c1 + c2 * c2 + c3 * c3 + c4 * c4) * 0.2 if mean is None else mean
    eps = eps_rel * m + 1e-300
    b0 = 13.0 / 12.0 * (c0 - 2 * c1 + c2) ** 2 + 0.25 * (c0 - 4 * c1 + 3 * c2) ** 2
    b1 = 13.0 / 12.0 * (c1 - 2 * c2 + c3) ** 2 + 0.25 * (c1 - c3) ** 2
    b2 = 13.0 / 12.0 * (c2 - 2 * c3 + c4) ** 2 + 0.25 * (3 * c2 - 4 * c3 + c4) ** 2
    tau = (b0 - b2).abs()
    return 0.1 * (1 + tau / (b0 + eps)), 0.6 * (1 + tau / (b1 + eps)), 0.3 * (1 + tau / (b2 + eps))


def _weno5(c, eps_rel=1e-6):
    c0, c1, c2, c3, c4 = c
    a0, a1, a2 = _weno5_weights(c, eps_rel)
    p0, p1, p2 = (2 * c0 - 7 * c1 + 11 * c2) / 6, (-c1 + 5 * c2 + 2 * c3) / 6, (2 * c2 + 5 * c3 - c4) / 6
    return (a0 * p0 + a1 * p1 + a2 * p2) / (a0 + a1 + a2)


def _weno3(c0, c1, c2, eps_rel=1e-6):
    eps = eps_rel * (c0 * c0 + c1 * c1 + c2 * c2) / 3 + 1e-300
    b0, b1 = (c1 - c0) ** 2, (c2 - c1) ** 2
    tau = (b0 - b1).abs()
    a0, a1 = (1 + tau / (b0 + eps)) / 3, 2 * (1 + tau / (b1 + eps)) / 3
    return (a0 * (-0.5 * c0 + 1.5 * c1) + a1 * (0.5 * c1 + 0.5 * c2)) / (a0 + a1)


def _slope(lim, a, b):
    ab = a * b
    if lim == "MC":
        m = torch.minimum(torch.minimum(2 * a.abs(), 0.5 * (a + b).abs()), 2 * b.abs())
        return torch.where(ab > 0, m * torch.sign(a), torch.zeros_like(a))
    s = torch.where(ab > 0, a + b, torch.ones_like(a))
    return torch.where(ab > 0, 2 * ab / s, torch.zeros_like(a))


def _face_values(recon, lim, c):
    """Left and right values from the six cells around the face."""
    if recon == "weno5":
        return _weno5(c[:5]), _weno5(c[:0:-1])
    if recon == "weno3":
        return _weno3(c[1], c[2], c[3]), _weno3(c[4], c[3], c[2])
    return c[2] + 0.5 * _slope(lim, c[2] - c[1], c[3] - c[2]), c[3] - 0.5 * _slope(lim, c[4] - c[3], c[3] - c[2])


class _Run:
    """One uniform run: state, residual, steps."""

    def __init__(self, case, U):
        k = _keys(case)
        self.k, self.gas = k, _Gas(float(k["gamma"]))
        self.n = [int(k["nx"]), int(k["ny"]), int(k["nz"])]
        self.nd = 3 if self.n[2] > 1 else 2
        L = [float(k["Lx"]), float(k["Ly"]), float(k.get("Lz", 1.0))]
        self.L, self.h = L, [L[a] / self.n[a] for a in range(3)]
        sides = ["xmin", "xmax", "ymin", "ymax", "zmin", "zmax"]
        self.bc = [str(k.get("bc_" + s, "periodic")) for s in sides]
        self.per = [self.bc[2 * a] == "periodic" and self.bc[2 * a + 1] == "periodic" for a in range(3)]
        self.bo2 = str(k.get("boundary_order", 2)) == "2"
        self.recon, self.lim = k["reconstruction"], k.get("muscl_limiter", "Van Leer")
        self.lowmach = "Mach" in k["riemann_solver"]
        self.visc = k["use_viscous"] == "true"
        if self.visc:
            self.mu = float(k["mu"])
            self.kc = self.mu * self.gas.g / (float(k["pr"]) * (self.gas.g - 1.0))
        self.fourth = k.get("flux_quadrature") == "fourth"
        self.learned = k.get("indicator") == "learned"
        if self.learned:
            self.net, self.kept, self.off, self.count = _Net(), [None] * 3, False, 0
        self.cfl = float(k["cfl"])
        h = self.h
        self.len = min(h[0], h[1]) if self.nd == 2 else 2.0 / (1 / h[0] + 1 / h[1] + 1 / h[2])
        shape = (self.n[2], self.n[1], self.n[0])
        T = torch.from_numpy(np.ascontiguousarray(U.T)).to(_device())
        self.U = [T[q].reshape(shape).clone() for q in range(T.shape[0])]
        if len(self.U) == 4:
            self.U.append(torch.zeros_like(self.U[0]))
        self.t, self.s, self.lagged = 0.0, 0.0, 0.0

    # -- boundary states --
    def ghost(self, side, Ui):
        bc, a = self.bc[side], side // 2
        if bc == "transmissive":
            return Ui
        W = self.gas.prim(Ui)
        k = self.k
        if bc == "wall":
            W[MOM[a]] = -W[MOM[a]]
        elif bc == "no_slip":
            for m in MOM:
                W[m] = -W[m]
        elif bc in ("moving_wall", "massflow_inlet"):
            ut = float(k["u_in"]) if bc == "moving_wall" else self.ut
            W[1], W[2], W[4] = 2 * ut - W[1], 2 * float(k.get("v_in", 0.0)) - W[2], -W[4]
        else:
            raise ValueError(bc)
        return self.gas.cons(W)

    def nonreflecting(self, side, U):
        """Ghosts of the boundary cells of a non-reflecting side: only the incoming acoustic wave differs."""
        a, s, g = side // 2, 1.0 if side & 1 else -1.0, self.gas
        W = g.prim([_cut(t, a, self.n[a] - 1 if side & 1 else 0, 1) for t in U])
        c = g.sound(W)
        un = s * W[MOM[a]]
        M = (un / c).clamp(-1.0, 1.0)
        K = 0.28 * c * (1 - M * M) / self.L[a]
        beta, T1 = M.abs(), torch.zeros_like(c)
        for b in range(self.nd):
            n = self.n[b]
            if b == a or n == 1:
                continue
            if self.per[b]:
                lo, hi, span = [t.roll(1, _dim(b)) for t in W], [t.roll(-1, _dim(b)) for t in W], 2.0
            else:
                lo = [torch.cat([_cut(t, b, 0, 1), _cut(t, b, 0, n - 1)], _dim(b)) for t in W]
                hi = [torch.cat([_cut(t, b, 1, n - 1), _cut(t, b, n - 1, 1)], _dim(b)) for t in W]
                sp = torch.full((n,), 2.0, dtype=torch.float64, device=c.device)
                sp[0] -= 1.0
                sp[-1] -= 1.0
                span = sp.view([n if d == _dim(b) else 1 for d in range(3)])
            ht, m = span * self.h[b], MOM[b]
            T1 = T1 + (W[m] * (hi[3] - lo[3]) + W[0] * c * c * (hi[m] - lo[m]) - W[0] * c * s * W[m] * (hi[MOM[a]] - lo[MOM[a]])) / ht
        dw = -self.h[a] * (K * (W[3] - float(self.k["p_out"])) - (1 - beta) * T1) / (c - un)
        G = list(W)
        G[3], G[MOM[a]], G[0] = W[3] + 0.5 * dw, W[MOM[a]] - s * dw / (2 * W[0] * c), W[0] + 0.5 * dw / (c * c)
        return g.cons([torch.where(M >= 1, W[q], G[q]) for q in range(5)])

    def edge(self, U, side):
        a = side // 2
        return [_cut(t, a, self.n[a] - 1 if side & 1 else 0, 1) for t in U]

    def outside(self, U, side):
        a = side // 2
        if self.bc[side] == "periodic":
            return self.edge(U, side ^ 1)
        if self.bc[side] == "nonreflecting":
            return self.nonreflecting(side, U)
        return self.ghost(side, self.edge(U, side))

    def halo(self, a):
        """What lies outside each side of an axis: 1 wrap, 2 ghost slab, 0 nothing."""
        deep = 3 if self.recon == "weno5" else 2
        if self.per[a] and self.n[a] >= deep:
            return 1, 1
        slab = [2 if self.bo2 and self.n[a] >= deep and self.bc[2 * a + i] not in ("periodic", "nonreflecting") else 0 for i in (0, 1)]
        return slab[0], slab[1]

    def pad(self, U, V, a, prim=True):
        """V (the primitives or the conservative state of U) with three layers on both sides of axis a."""
        kinds, n, d = self.halo(a), self.n[a], _dim(a)
        out = []
        side_layers = []
        for i in (0, 1):
            if kinds[i] == 1:
                side_layers.append([_cut(t, a, n - 3 if i == 0 else 0, 3) for t in V])
            elif kinds[i] == 2:
                m = min(3, n)
                g = self.ghost(2 * a + i, [_cut(t, a, 0 if i == 0 else n - m, m).flip(d) for t in U])
                g = self.gas.prim(g) if prim else g
                if m < 3:
                    g = [torch.cat([t] + [_cut(t, a, m - 1, 1)] * (3 - m), d) if i else torch.cat([_cut(t, a, 0, 1)] * (3 - m) + [t], d)
                         for t in g]
                side_layers.append(g)
            else:
                side_layers.append([torch.cat([_cut(t, a, 0 if i == 0 else n - 1, 1)] * 3, d) for t in V])
        for q in range(5):
            out.append(torch.cat([side_layers[0][q], V[q], side_layers[1][q]], d))
        return out

    # -- viscous term --
    def visc_ghost(self, side, C):
        bc, a = self.bc[side], side // 2
        G = list(C)
        if bc == "no_slip":
            for m in MOM:
                G[m] = -C[m]
        elif bc == "wall":
            G[MOM[a]] = -C[MOM[a]]
        elif bc == "moving_wall":
            vel = (float(self.k["u_in"]), float(self.k.get("v_in", 0.0)), 0.0)
            for b in range(3):
                G[MOM[b]] = -C[MOM[b]] if b == a else 2 * C[0] * vel[b] - C[MOM[b]]
            if self.bo2:
                G[3] = C[3] + 0.5 * (G[1] ** 2 + G[2] ** 2 + G[4] ** 2 - C[1] ** 2 - C[2] ** 2 - C[4] ** 2) / C[0]
        return G

    def visc_pad(self, U):
        """One layer on every side, axis after axis, so that edges take the rule of the lower axis over the higher's."""
        P = list(U)
        for a in reversed(range(self.nd)):
            n = self.n[a]
            lo, hi = [_cut(t, a, 0, 1) for t in P], [_cut(t, a, n - 1, 1) for t in P]
            gl = hi if self.bc[2 * a] == "periodic" else self.visc_ghost(2 * a, lo)
            gh = lo if self.bc[2 * a + 1] == "periodic" else self.visc_ghost(2 * a + 1, hi)
            P = [torch.cat([gl[q], P[q], gh[q]], _dim(a)) for q in range(5)]
        return P

    def inner(self, t, skip=()):
        """A padded array without its layers, except along the axes in skip."""
        for a in range(self.nd):
            if a not in skip:
                t = _cut(t, a, 1, self.n[a])
        return t

    def viscous(self, U):
        """Per axis the viscous face fluxes (rho u, rho v, rho E, rho w) without the area, and the speed bound."""
        nd, h, P = self.nd, self.h, self.visc_pad(U)
        PW = self.gas.prim(P)
        W = self.gas.prim(U)
        grad = {}
        for b in range(nd):
            d = [(_cut(self.inner(P[q], (b,)), b, 2, self.n[b]) - _cut(self.inner(P[q], (b,)), b, 0, self.n[b])) / (2 * h[b]) for q in range(5)]
            for i in range(nd):
                grad[i, b] = (d[MOM[i]] - W[MOM[i]] * d[0]) / W[0]
        inv_h2 = sum(1 / h[a] ** 2 for a in range(nd))
        nu = torch.maximum(4.0 / 3.0 * self.mu / W[0], self.kc * (self.gas.g - 1) / W[0]) + 1e-12
        vmax = torch.stack([W[MOM[a]].abs() for a in range(nd)]).amax(0)
        bound = float((vmax + self.gas.sound(W) + 2 * self.len * inv_h2 * nu).max())
        fluxes = []
        for a in range(nd):
            n, d = self.n[a], _dim(a)
            line = [self.inner(t, (a,)) for t in PW]
            T = line[3] / line[0]
            left = lambda t: _cut(t, a, 0, n + 1)   # noqa: E731
            right = lambda t: _cut(t, a, 1, n + 1)   # noqa: E731
            gn = [(right(line[MOM[i]]) - left(line[MOM[i]])) / h[a] for i in range(nd)]
            vf = [0.5 * (right(line[MOM[i]]) + left(line[MOM[i]])) for i in range(nd)]
            dT = (right(T) - left(T)) / h[a]

            def cross(i, b):
                g = grad[i, b]
                lo, hi = _cut(g, a, 0, 1), _cut(g, a, n - 1, 1)
                gl = torch.cat([hi if self.per[a] else lo, g], d)
                gr = torch.cat([g, lo if self.per[a] else hi], d)
                c = 0.5 * (gl + gr)
                if self.bo2 and not self.per[a]:   # tangential difference of the face velocity on the boundary faces
                    wide = self.inner(PW[MOM[i]], (a, b))
                    for at, pair in ((0, (0, 1)), (n, (n, n + 1))):
                        f = 0.5 * (_cut(wide, a, pair[0], 1) + _cut(wide, a, pair[1], 1))
                        _cut(c, a, at, 1).copy_((_cut(f, b, 2, self.n[b]) - _cut(f, b, 0, self.n[b])) / (2 * h[b]))
                return c

            others = [b for b in range(nd) if b != a]
            div = sum(cross(b, b) for b in others)
            tau = [None] * 3
            tau[a] = self.mu * (4.0 / 3.0 * gn[a] - 2.0 / 3.0 * div)
            for b in others:
                tau[b] = self.mu * (gn[b] + cross(a, b))
            en = sum(vf[i] * tau[i] for i in range(nd)) + self.kc * dT
            fluxes.append([torch.zeros_like(en), tau[0], tau[1], en, tau[2] if nd == 3 else torch.zeros_like(en)])
        return fluxes, bound

    # -- convective faces --
    def face_states(self, U, W, a, predictor=None):
        n, d = self.n[a], _dim(a)
        if predictor is not None:   # MUSCL-Hancock on a periodic axis: the neighbours' advanced states
            lo, hi = predictor[2 * a], predictor[2 * a + 1]
            UL = [torch.cat([_cut(t, a, n - 1, 1), t], d) for t in hi]
            UR = [torch.cat([t, _cut(t, a, 0, 1)], d) for t in lo]
            return UL, UR
        P = self.pad(U, W, a)
        wl, wr = [], []
        smooth = self.smooth_faces(P, a) if self.learned else None
        for q in range(5):
            c = [_cut(P[q], a, s, n + 1) for s in range(6)]
            x, y = _face_values(self.recon, self.lim, c)
            if smooth is not None:
                up = lambda c0, c1, c2, c3, c4: (2 * c0 - 13 * c1 + 47 * c2 + 27 * c3 - 3 * c4) / 60   # noqa: E731
                x, y = torch.where(smooth, up(*c[:5]), x), torch.where(smooth, up(*c[:0:-1]), y)
            wl.append(x)
            wr.append(y)
        UL, UR = self.gas.cons(wl), self.gas.cons(wr)
        for i, kind in enumerate(self.halo(a)):
            if kind:
                continue
            side, at = 2 * a + i, n if i else 0   # a side face without a full stencil: the first-order states
            out, cell = self.outside(U, side), self.edge(U, side)
            out, cell = self.gas.cons(self.gas.prim(out)), self.gas.cons(self.gas.prim(cell))
            for q in range(5):
                _cut(UL[q], a, at, 1).copy_(cell[q] if i else out[q])
                _cut(UR[q], a, at, 1).copy_(out[q] if i else cell[q])
        return UL, UR

    def smooth_faces(self, P, a):
        """The network's decision on the faces of a periodic axis, kept from the step's first stage."""
        if self.off:
            return None
        if self.stage == 1:
            n = self.n[a]
            c = [[_cut(P[q], a, s, n + 1) for s in range(6)] for q in range(5)]
            self.kept[a] = self.net.troubled(c)
            if self.count % 50 == 0:
                label = self.net.label(c) > 0.05
                hit = self.kept[a]
                self.audit += torch.stack([(label & hit).sum(), (~label & hit).sum(), (label & ~hit).sum(), (~label & ~hit).sum()])
        return ~self.kept[a]

    def predict(self, U, W, half):
        """The limited states of every cell (low and high face of each axis) advanced by half a step."""
        st, dd = [], [0.0] * 5
        for a in range(self.nd):
            P = self.pad(U, W, a)
            n = self.n[a]
            lo, hi = [], []
            for q in range(5):
                m, z, p = (_cut(P[q], a, s, n) for s in (2, 3, 4))
                lo.append(z - 0.5 * _slope(self.lim, p - z, z - m))
                hi.append(z + 0.5 * _slope(self.lim, z - m, p - z))
            pair = [self.gas.cons(lo), self.gas.cons(hi)]
            st += pair
            f = []
            for S in pair:
                w = self.gas.prim(S)
                F = [S[0] * w[MOM[a]], S[1] * w[MOM[a]], S[2] * w[MOM[a]], (S[3] + w[3]) * w[MOM[a]], S[4] * w[MOM[a]]]
                F[MOM[a]] = F[MOM[a]] + w[3]
                f.append(F)
            dd = [dd[q] + half / self.h[a] * (f[1][q] - f[0][q]) for q in range(5)]
        out = []
        for S in st:
            N = [S[q] - dd[q] for q in range(5)]
            ok = (N[0] > 1e-10) & (0.5 * (N[1] ** 2 + N[2] ** 2 + N[4] ** 2) < N[0] * N[3])
            out.append([torch.where(ok, N[q], S[q]) for q in range(5)])
        return out

    def fourth_fluxes(self, U, a):
        """Fluxes of the faces of a periodic axis with the fourth-order quadrature, and the largest wave speed."""
        n, d, g1 = self.n[a], _dim(a), self.gas.g - 1.0
        P = self.pad(U, U, a, prim=False)
        c = [[_cut(P[q], a, s, n + 1) for q in range(5)] for s in range(6)]
        ul, ur = [], []
        for q in range(5):
            x, y = _face_values(self.recon, self.lim, [c[s][q] for s in range(6)])
            ul.append(x)
            ur.append(y)
        m2 = lambda u: u[1] ** 2 + u[2] ** 2 + u[4] ** 2   # noqa: E731
        positive = lambda u: (u[0] > 0) & (g1 * (u[3] * u[0] - 0.5 * m2(u)) > 0)   # noqa: E731
        pressure = lambda u: g1 * (u[3] - 0.5 * m2(u) / u[0])   # noqa: E731
        cp = torch.stack([pressure(u) for u in c])
        cr = torch.stack([u[0] for u in c])
        ok = positive(ul) & positive(ur)
        for v, lo, hi in ((cr, cr.amin(0), cr.amax(0)), (cp, cp.amin(0), cp.amax(0))):
            wide = hi - lo
            for u in (ul, ur):
                t = u[0] if v is cr else pressure(u)
                ok = ok & (t >= lo - wide) & (t <= hi + wide)
        ul = [torch.where(ok, ul[q], c[2][q]) for q in range(5)]
        ur = [torch.where(ok, ur[q], c[3][q]) for q in range(5)]
        pl, pr = pressure(ul), pressure(ur)
        good = positive(ul) & positive(ur) & ((pr - pl).abs() <= 0.2 * torch.minimum(pl, pr))
        trans = [b for b in range(self.nd) if b != a]

        def all_nbrs(m):
            out = m
            for b in trans:
                out = out & m.roll(1, _dim(b)) & m.roll(-1, _dim(b))
            return out

        def lap(t):
            return sum(t.roll(1, _dim(b)) - 2 * t + t.roll(-1, _dim(b)) for b in trans)

        al, ar = [t - lap(t) / 24 for t in ul], [t - lap(t) / 24 for t in ur]
        pt = all_nbrs(good) & positive(al) & positive(ar)
        al = [torch.where(pt, al[q], ul[q]) for q in range(5)]
        ar = [torch.where(pt, ar[q], ur[q]) for q in range(5)]
        Fp, s = _hllc(self.gas, al, ar, a, self.lowmach)
        F0, _ = _hllc(self.gas, ul, ur, a, self.lowmach)
        full = all_nbrs(pt)
        return [torch.where(full, Fp[q] + lap(Fp[q]) / 24, torch.where(pt, F0[q], Fp[q])) for q in range(5)], s

    def residual(self, U, half=0.0):
        W = self.gas.prim(U)
        for side in range(2 * self.nd):
            if self.bc[side] == "massflow_inlet":
                rho = float(self.edge(U, side)[0].clamp_min(1e-10).mean())
                self.ut = float(self.k["rho_in"]) * float(self.k["u_in"]) / max(rho, 1e-5)
        pred = self.predict(U, W, half) if half > 0 else None
        R, S = [0.0] * 5, 0.0
        for a in range(self.nd):
            n = self.n[a]
            if self.fourth:
                F, s = self.fourth_fluxes(U, a)
            else:
                UL, UR = self.face_states(U, W, a, pred)
                F, s = _hllc(self.gas, UL, UR, a, self.lowmach)
                del UL, UR
            S = max(S, s)
            R = [R[q] - (_cut(F[q], a, 1, n) - _cut(F[q], a, 0, n)) / self.h[a] for q in range(5)]
        if self.visc:
            V, bound = self.viscous(U)
            S = max(S, bound)
            for a in range(self.nd):
                n = self.n[a]
                R = [R[q] + (_cut(V[a][q], a, 1, n) - _cut(V[a][q], a, 0, n)) / self.h[a] for q in range(5)]
        return R, S

    def step(self, t_max=FAR):
        U, scheme = self.U, self.k["time_scheme"]

        def dt_of(S):
            return min(self.cfl * self.len / (S + 1e-10), t_max - self.t)

        if scheme == "MUSCL-Hancock":
            if self.lagged <= 0:
                self.lagged = self.residual(U)[1]
            dt = dt_of(self.lagged)
            R, S = self.residual(U, 0.5 * dt)
            self.U, self.lagged, self.s = [U[q] + dt * R[q] for q in range(5)], S, S
            self.t += dt
            return
        self.stage, self.audit = 1, torch.zeros(4, dtype=torch.int64, device=U[0].device)
        R, S = self.residual(U)
        dt = dt_of(S)
        V = [U[q] + dt * R[q] for q in range(5)]
        self.stage = 2
        R, s2 = self.residual(V)
        if scheme.endswith("2"):
            self.U, self.s = [0.5 * U[q] + 0.5 * (V[q] + dt * R[q]) for q in range(5)], max(S, s2)
        else:
            V = [0.75 * U[q] + 0.25 * (V[q] + dt * R[q]) for q in range(5)]
            R, s3 = self.residual(V)
            self.U, self.s = [U[q] / 3 + 2 * (V[q] + dt * R[q]) / 3 for q in range(5)], max(S, s2, s3)
        self.t += dt
        if self.learned:
            tp, fp, fn, tn = (float(v) for v in self.audit)
            if self.count % 50 == 0 and not self.off and tp + fn > 0 and fn > 0.01 * (tp + fn) and fn > 1e-4 * (tp + fp + fn + tn):
                self.off = True
            self.count += 1

    def cells(self, V, ncomp):
        return torch.stack([t.reshape(-1) for t in V[:ncomp]], dim=1)

    def monitor(self):
        self.stage = 1
        R, _ = self.residual(self.U)
        U = self.U
        ke = 0.5 * (U[1] ** 2 + U[2] ** 2 + U[4] ** 2) / U[0]
        rms = lambda t: float(torch.sqrt(t.mean()))   # noqa: E731
        return np.array([float(U[0].mean()), float(ke.mean()), float(U[3].mean()), rms(R[0] ** 2), rms(R[1] ** 2 + R[2] ** 2 + R[4] ** 2),
                         rms(R[3] ** 2)])


class _Net:
    """The indicator's features, network and label on six-cell stencils (three velocity components)."""

    def __init__(self):
        p, thr = _weights()
        p = torch.from_numpy(np.asarray(p)).to(_device())
        self.W1, self.b1, self.W2 = p[:480].view(32, 15), p[480:512], p[512:1536].view(32, 32)
        self.b2, self.w3, self.b3, self.thr = p[1536:1568], p[1568:1600], p[1600], thr

    def troubled(self, c):
        c = [[t.float() for t in v] for v in c]
        tv = torch.stack([sum((v[j + 1] - v[j]).abs() for j in range(5)) for v in (c[1], c[2], c[4])]).argmax(0)
        vel = [torch.where(tv == 0, c[1][j], torch.where(tv == 1, c[2][j], c[4][j])) for j in range(6)]
        x = []
        for v in (c[0], c[3], vel):
            d = [v[j + 1] - v[j] for j in range(5)]
            norm = torch.sqrt(sum(t * t for t in d) + 1e-6 * sum(t * t for t in v) / 6 + 1e-30)
            x += [(d[j + 1] - d[j]) / norm for j in range(4)] + [torch.stack([t.abs() for t in d]).amax(0) / norm]
        X = torch.stack([t.reshape(-1) for t in x], dim=1)
        out = []
        r = lambda t: t.bfloat16().float()   # noqa: E731
        for part in X.split(1 << 21):
            h = r((r(part) @ r(self.W1).T + r(self.b1)).clamp_min(0))
            h = (h @ r(self.W2).T + self.b2).clamp_min(0)
            out.append(h @ self.w3 + self.b3 > self.thr)
        return torch.cat(out).view(c[0][0].shape)

    def label(self, c):
        scale = sum(c[1][j] ** 2 + c[2][j] ** 2 + c[4][j] ** 2 + c[3][j] / c[0][j] for j in range(6)) / 6
        out = torch.zeros_like(scale)
        for q in range(5):
            for s in (c[q][:5], c[q][:0:-1]):
                w = _weno5_weights(s, 1e-6, scale if q in MOM else None)
                tot = w[0] + w[1] + w[2]
                for k, lin in enumerate((0.1, 0.6, 0.3)):
                    out = torch.maximum(out, (w[k] / tot - lin).abs())
        return out


def _exact_riemann(case, n, U):
    """The 1-D ensemble with all instances side by side: rows of the longest length, each with its own time and step."""
    d, g = _device(), _Gas(1.4)
    ninst, N = len(n), int(max(n))
    nn = torch.tensor(np.asarray(n), dtype=torch.int64, device=d).view(-1, 1)
    off = np.concatenate([[0], np.cumsum(n)])
    V = torch.zeros(5, ninst, N, dtype=torch.float64, device=d)
    V[0], V[3] = 1.0, 1.0
    T = torch.from_numpy(np.ascontiguousarray(U.T)).to(d)
    for i in range(ninst):
        V[0, i, :n[i]], V[1, i, :n[i]], V[3, i, :n[i]] = (T[q, off[i]:off[i + 1]] for q in (0, 1, 3))
    j = torch.arange(-2, N + 3, device=d).view(1, -1)   # the ghost slab of a transmissive end mirrors the cells
    at = torch.where(j < 0, -1 - j, torch.where(j >= nn, 2 * nn - 1 - j, j)).clamp(0, N - 1)
    face = torch.arange(N + 1, device=d).view(1, -1) <= nn
    cell = torch.arange(N, device=d).view(1, -1) < nn
    h = 1.0 / nn.double()

    def residual(V):
        W = torch.stack(g.prim(list(V)))
        S = torch.where(cell, W[2].abs() + g.sound(list(W)), torch.zeros_like(W[0])).amax(1)
        P = W[:, torch.arange(ninst, device=d).view(-1, 1), at]
        wl, wr = [], []
        for q in range(5):
            c = [P[q][:, s:s + N + 1] for s in range(4)]
            wl.append(c[1] + 0.5 * _slope("MC", c[1] - c[0], c[2] - c[1]))
            wr.append(c[2] - 0.5 * _slope("MC", c[3] - c[2], c[2] - c[1]))
        for w in (wl, wr):   # faces beyond an instance's end: any admissible state
            for q in (0, 3):
                w[q] = torch.where(face, w[q], torch.ones_like(w[q]))
        UL, UR = g.cons(wl), g.cons(wr)
        F, _ = _hllc(g, UL, UR, 0, False)
        WL, WR = g.prim(UL), g.prim(UR)
        cl, cr = g.sound(WL), g.sound(WR)
        s = torch.maximum(torch.minimum(WL[1] - cl, WR[1] - cr).abs(), torch.maximum(WL[1] + cl, WR[1] + cr).abs())
        S = torch.maximum(S, torch.where(face, s, torch.zeros_like(s)).amax(1))
        F = torch.stack(F)
        return torch.where(cell, -(F[:, :, 1:] - F[:, :, :-1]) / h, torch.zeros_like(V)), S.view(-1, 1)

    t = torch.zeros(ninst, 1, dtype=torch.float64, device=d)
    steps, last = torch.zeros_like(nn), torch.zeros_like(t)
    while True:
        live = t < case["t_end"]
        if not bool(live.any()):
            break
        R, s1 = residual(V)
        dt = torch.minimum(0.5 * h / (s1 + 1e-10), case["t_end"] - t)
        A = V + dt * R
        R, s2 = residual(A)
        V = torch.where(live, 0.5 * V + 0.5 * (A + dt * R), V)
        t = torch.where(live, t + dt, t)
        steps += live
        last = torch.where(live, torch.maximum(s1, s2), last)
    out = torch.cat([V[:, i, :n[i]] for i in range(ninst)], dim=1)
    return dict(U=torch.stack([out[0], out[1], out[3]], dim=1), t=t.view(-1), steps=None, s=last.view(-1))


def exact(case, seed):
    f = case["family"]
    if f == "riemann":
        n, U = _flow(case, seed)
        # steps of the longest run, from the initial wave speeds (they grow by up to about two), at 1.5 ms a step
        o = np.concatenate([[0], np.cumsum(n)])
        p = 0.4 * (U[:, 3] - 0.5 * U[:, 1] ** 2 / U[:, 0])
        s = np.abs(U[:, 1] / U[:, 0]) + np.sqrt(1.4 * p / U[:, 0])
        if max(2.0 * case["t_end"] * s[o[i]:o[i + 1]].max() * n[i] / 0.5 for i in range(len(n))) > 5000:
            return None
        return _exact_riemann(case, n, U)
    if f == "vortices":
        n, U = _flow(case, seed)
        if sum(case["t_end"] * 3.0 * int(k) / 10.0 / 0.5 for k in n) > 2400:   # about 8 ms a step
            return None
        off, outs, ts, ss = np.concatenate([[0], np.cumsum(n.astype(np.int64) ** 2)]), [], [], []
        for i, k in enumerate(n):
            u = U[off[i]:off[i + 1]]
            r = _Run(dict(case, nx=int(k), ny=int(k)), u)
            while r.t < case["t_end"]:
                r.step(case["t_end"])
            outs.append(r.cells(r.U, 4))
            ts.append(r.t)
            ss.append(r.s)
        return dict(U=torch.cat(outs), t=np.array(ts), steps=None, s=np.array(ss))
    nz = case.get("nz", 1)
    stages = 3 * case.get("steps", 1)
    if case["nx"] * case["ny"] * nz * stages * 1.5e-8 * (2.0 if case.get("quad") == "fourth" else 1.0) > 18.0:
        return None
    U = _flow(case, seed)
    r = _Run(case, U)
    if f == "residual":
        R, s = r.residual(r.U)
        return dict(R=r.cells(R, U.shape[1]), s=s)
    for _ in range(case["steps"]):
        r.step()
    out = dict(U=r.cells(r.U, U.shape[1]), t=r.t, s=r.s)
    if case.get("monitor"):
        out["monitor"] = r.monitor()
    return out
