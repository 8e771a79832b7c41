"""Timed workloads of the RK3 dynamical core, through the calls a host model or a torch
harness makes (olam_amd.gpu.Context, olam_amd.adjoint.transport).

A case is a dict of plain values; ``prepare`` builds the context and its seeded inputs,
``run`` makes one pass and ``exact`` evaluates the same pass in 64-bit torch from the
formulas of the model (no kernel or oracle of this package).  Grids, the jet state and the
prescribed winds depend on the grid only and are kept per process; the tracers, the
adjoint fields, the warm anomaly and the tendencies are drawn from the seed.

Kinds of pass:
  acoustic   tend0 and one prog_wrtv_rk; a host coupling the acoustic step to its physics
  tracer     one scalar_transport_rk with prescribed winds, tracers in and out as tensors
  gradient   the same step and its adjoint, as one layer of a gradient computation
  longstep   tend0, nacoust x prog_wrtv_rk, timeavg_momsc, scalar_transport_rk and, with
             ``adjoint``, its adjoint; with ``physics`` the host's PBL and moisture fields
             are set before it, as its namelist does every long step
  window     a multi-step window with checkpoints, forward and backward, under autograd
  host       one long step of a host whose arrays live in host memory: tendencies up,
             the fields its physics reads and the tracers down
  diagnose   mass sums, tracer extrema and the CFL report of a history step
"""

from __future__ import annotations

import functools
import math

import numpy as np
import torch

from olam_amd import abi, cases as C, mesh as M
from olam_amd.adjoint import TransportWindow, transport
from olam_amd.gpu import Context

DEV = "cuda" if torch.cuda.is_available() else "cpu"
RAYF = {"rayf": (27000.0, 0.0, 1.0), "rayfw": (27000.0, 0.5, 1.0),
        "rayfdiv": (27000.0, 0.15, 1.0), "rayfmix": (27000.0, 0.25, 1.0)}
DEFAULTS = dict(ntr=0, prec="f32", order=2, nrk_scal=3, monot=0, mono_dyn=0, nacoust=1, adjoint=False,
                physics=False, nsteps=1)


def _case(name, kind, nxp, nlev, **kw):
    c = dict(DEFAULTS, kind=kind, nxp=nxp, nlev=nlev, **kw)
    return dict(c, name=name) if name else c


def listed():
    return [
        # the smallest call there is: a coarse test run, all launches and latency
        _case("acoustic_nxp8_L16_f32", "acoustic", 8, 16),
        # a single-tracer advection test in 64 bits (cosine-bell class of runs)
        _case("tracer_nxp40_L30_f64_1", "tracer", 40, 30, ntr=1, prec="f64"),
        # the regional-resolution dry dynamics in the reference's own precision
        _case("acoustic_nxp160_L50_mixed", "acoustic", 160, 50, prec="mixed"),
        # one step of a 4-tracer inversion: forward and gradient
        _case("gradient_nxp160_L50_4", "gradient", 160, 50, ntr=4),
        # the production step: dynamics, 10 tracers and their adjoint on a million columns
        _case("longstep_nxp320_L60_10", "longstep", 320, 60, ntr=10, adjoint=True),
        # the reference's test namelist: 3 acoustic steps, RK2 tracers, PBL, moisture, friction
        _case("namelist_nxp40_L45_3", "longstep", 40, 45, ntr=3, nrk_scal=2, nacoust=3, physics=True),
        # chemistry-like tracers that must not over- or undershoot
        _case("monotone_nxp64_L41_5", "tracer", 64, 41, ntr=5, monot=1),
        # deep columns (two wavefronts each), many tracers, forward and gradient
        _case("gradient_nxp64_L70_20", "gradient", 64, 70, ntr=20),
        # third-order reconstruction, forward and gradient
        _case("order3_nxp48_L60_8", "gradient", 48, 60, ntr=8, order=3),
        # drop-in host: everything its physics touches crosses PCIe every step
        _case("host_nxp64_L60_10", "host", 64, 60, ntr=10),
        # a history step's diagnostics
        _case("diagnose_nxp160_L50_10", "diagnose", 160, 50, ntr=10),
        # a 4-step window with checkpoints under autograd
        _case("window_nxp64_L50_4", "window", 64, 50, ntr=4, nsteps=4),
    ]


def draw(rng):
    kind = rng.choice(["acoustic", "acoustic", "tracer", "tracer", "gradient", "gradient", "longstep", "host",
                       "diagnose", "window"])
    while True:
        nxp = int(round(math.exp(rng.uniform(math.log(8), math.log(140)))))
        nlev = rng.choice([rng.randint(10, 63), rng.randint(30, 63), rng.randint(64, 90)])
        ntr = 0 if kind == "acoustic" else int(round(math.exp(rng.uniform(0.0, math.log(24)))))
        if (10 * nxp * nxp + 2) * nlev * (8 + ntr) < 1.0e8:
            break
    kw = dict(ntr=ntr, prec=rng.choice(["f32", "f32", "f32", "mixed", "f64"]), order=rng.choice([2, 2, 2, 2, 1, 3]))
    if kind in ("tracer", "gradient"):
        kw.update(monot=rng.choice([0, 0, 0, 1, 2]), nrk_scal=rng.choice([3, 3, 2]))
    if kind == "acoustic":
        kw.update(mono_dyn=rng.choice([0, 0, 0, 1]))
    if kind == "longstep":
        kw.update(adjoint=rng.choice([True, False]), nacoust=rng.choice([1, 2, 3]))
    if kind == "window":
        kw.update(nsteps=rng.randint(2, 6))
    return _case(None, kind, nxp, nlev, **kw)


# ------------------------------------------------------------------ what depends on the grid
@functools.lru_cache(maxsize=None)
def _grid(nxp, nlev):
    return abi.FortranGrid(M.build_mesh(nxp), M.vertical_grid(nlev))


@functools.lru_cache(maxsize=None)
def _jet(nxp, nlev):
    return C.jet_state(_grid(nxp, nlev))


@functools.lru_cache(maxsize=None)
def _winds(nxp, nlev):
    return C.transport_winds(_grid(nxp, nlev), _dt(nxp))


def _dt(nxp):
    """The step in use at 45 km and finer scaled with the cell size, a minute at most."""
    return min(60.0, 9600.0 / nxp)


def _params(case):
    dt = _dt(case["nxp"]) / case["nacoust"]
    return abi.make_params(case["prec"], num_scalar=case["ntr"], nrk_scal=case["nrk_scal"], order=case["order"],
                           iscal_monot=case["monot"], ithil_monot=case["mono_dyn"], iwind_monot=case["mono_dyn"],
                           dtsm=dt, dtlm=dt * case["nacoust"], nacoust=case["nacoust"],
                           initial=2 if case["physics"] else 1, rayf=RAYF if case["physics"] else None,
                           divh_damp_fact=0.12 if case["physics"] else 0.1)


# ------------------------------------------------------------------ seeded inputs
def _gen(seed, stream):
    return torch.Generator(device=DEV).manual_seed(int(seed) * 1009 + stream)


def _normal(grid, seed, stream, dtype, scale=1.0):
    z = torch.randn((grid.mwa - 1, grid.mza), generator=_gen(seed, stream), device=DEV, dtype=torch.float32)
    return (z * scale).to(dtype)


def _tracers(case, seed, dtype):
    """ln q ~ N(-20, 2) per cell-level, (ntr, N_W, mza)."""
    g = _grid(case["nxp"], case["nlev"])
    q = torch.empty((case["ntr"], g.mwa - 1, g.mza), dtype=dtype, device=DEV)
    for n in range(case["ntr"]):
        q[n] = torch.exp(-20.0 + 2.0 * _normal(g, seed, n, torch.float32)).to(dtype)
    q[:, :, 0] = q[:, :, 1]
    return q


def _adjoints(case, seed, dtype):
    """dJ/dq of a sum of random weights, (ntr, N_W, mza); nothing below the ground."""
    g = _grid(case["nxp"], case["nlev"])
    lam = torch.empty((case["ntr"], g.mwa - 1, g.mza), dtype=dtype, device=DEV)
    for n in range(case["ntr"]):
        lam[n] = _normal(g, seed, 100 + n, dtype)
    lam[:, :, 0] = 0
    return lam


def _anomaly(case, seed):
    """thil and rho (N_W, mza; FP64) of the jet state with a seeded warm anomaly of 1 K at
    unchanged pressure."""
    g = _grid(case["nxp"], case["nlev"])
    st = _jet(case["nxp"], case["nlev"]).arrays
    th = torch.from_numpy(st["thil"][1:]).to(DEV).double()
    rho = torch.from_numpy(st["rho"][1:]).to(DEV)
    rng = np.random.default_rng(seed)
    lat, lon = math.radians(rng.uniform(-60, 60)), rng.uniform(0, 2 * math.pi)
    at = torch.tensor([math.cos(lat) * math.cos(lon), math.cos(lat) * math.sin(lon), math.sin(lat)], device=DEV,
                      dtype=torch.float64)
    xyz = torch.stack([torch.from_numpy(g.arrays[n][1:]).to(DEV).double() for n in ("wnx", "wny", "wnz")], 1)
    r = M.ERAD * torch.acos((xyz @ at).clamp(-1, 1))
    zt = torch.from_numpy(g.arrays["zt"]).to(DEV).double()
    th1 = th + torch.exp(-(r / 1.5e6) ** 2)[:, None] * torch.exp(-((zt - 5000.0) / 2000.0) ** 2)[None, :]
    th1 = th1.float().double()
    return th1, rho * th / th1


def _tendencies(case, seed):
    """What a host's physics adds per unit volume: a heating of about a K per day, a drag of
    about a m/s per day and a percent of the tracer per hour (host arrays)."""
    g = _grid(case["nxp"], case["nlev"])
    rng = np.random.default_rng(seed + 77)

    def f(n, scale):
        a = np.zeros((n, g.mza), np.float32)
        a[1:, 1:] = rng.standard_normal((n - 1, g.mza - 1), dtype=np.float32) * np.float32(scale)
        return a

    st = {n: f(g.mwa, s) for n, s in (("thilt", 1e-5), ("vmxet", 1e-5), ("vmyet", 1e-5), ("vmzet", 1e-5))}
    st["vmt"] = np.zeros((g.mva, g.mza), np.float32)
    return st, [f(g.mwa, 1e-8 * 2.8e-6) for _ in range(case["ntr"])]


def _physics(case, seed):
    """PBL diffusivities below seeded tops, a surface drag, and moisture of the lower levels."""
    g = _grid(case["nxp"], case["nlev"])
    rng = np.random.default_rng(seed + 5)
    shape = (g.mwa, g.mza)
    top = max(3, g.mza // 3)
    turb = (rng.uniform(5.0, 100.0, shape).astype(np.float32), rng.uniform(5.0, 100.0, shape).astype(np.float32),
            rng.integers(2, top, g.mwa).astype(np.int32), rng.integers(2, top, g.mwa).astype(np.int32),
            np.full(g.mwa, 1e-3, np.float32) * g.arrays["arw0"])
    moist = np.exp(-g.arrays["zt"] / 2500.0)[None, :]
    rv = (moist * rng.uniform(0.004, 0.015, shape)).astype(np.float32)
    rw = (rv * rng.uniform(1.0, 1.1, shape)).astype(np.float32)
    theta = (_jet(case["nxp"], case["nlev"]).arrays["thil"] * rng.uniform(1.0, 1.005, shape)).astype(np.float32)
    return turb, (rv, rw, theta)


# ------------------------------------------------------------------ prepare and run
def _real(case):
    return torch.float64 if case["prec"] == "f64" else torch.float32


def _field(ctx, name, index=0):
    """A device tensor of one field's size and type."""
    f64 = ctx.params.precision == 2 or (name in ("rho", "press") and ctx.params.precision == 1)
    n = (ctx.grid.mva if name in ("vmc", "vmasc") else ctx.grid.mwa) - 1
    return torch.empty((n, ctx.grid.mza), dtype=torch.float64 if f64 else torch.float32, device=DEV)


def _put(ctx, name, t, index=0):
    ctx.copy_field(name, index, t.data_ptr(), 1)


def _put_all(ctx, name, q):
    for n in range(q.shape[0]):
        _put(ctx, name, q[n], n + 1)


def _get_all(ctx, name, out):
    for n in range(out.shape[0]):
        ctx.copy_field(name, n + 1, out[n].data_ptr(), 0)


def prepare(case, seed):
    grid = _grid(case["nxp"], case["nlev"])
    ctx = Context(grid, _params(case), device=0)
    kind, real = case["kind"], _real(case)
    s = {"case": case, "ctx": ctx}
    if kind in ("tracer", "gradient", "diagnose"):
        w = _winds(case["nxp"], case["nlev"])
        st = abi.FortranState.__new__(abi.FortranState)
        st.grid, st.arrays = grid, {n: w[n] for n in ("vmasc", "wmasc", "rho")}
        ctx.upload_state(st, only=("vmasc", "wmasc", "rho"))
        ro = torch.from_numpy(w["rho_old"][1:]).to(DEV, real).contiguous()
        torch.cuda.synchronize()
        _put(ctx, "rho_old", ro)
    else:
        ctx.upload_state(_jet(case["nxp"], case["nlev"]))
        th, rho = _anomaly(case, seed)
        th, rho = th.to(_field(ctx, "thil").dtype), rho.to(_field(ctx, "rho").dtype)
        torch.cuda.synchronize()
        _put(ctx, "thil", th)
        _put(ctx, "rho", rho)
        ctx.init_wrtv_rk()
        s["fields"] = {n: _field(ctx, n) for n in ("thil", "rho", "press", "wmc", "vmc")}
    if case["ntr"]:
        s["q"] = _tracers(case, seed, real)
        s["q_out"] = torch.empty_like(s["q"])
        if kind in ("gradient", "window") or case["adjoint"]:
            s["lam"] = _adjoints(case, seed, real)
            s["lam_out"] = torch.empty_like(s["lam"])
        torch.cuda.synchronize()
        if kind in ("longstep", "diagnose", "host"):
            _put_all(ctx, "scalar", s["q"])
        if kind == "longstep" and case["adjoint"]:
            _put_all(ctx, "scalar_adj", s["lam"])
    if kind == "host":
        tend, s["sct"] = _tendencies(case, seed)
        s["up"] = abi.FortranState(grid, tend)
        s["down"] = abi.FortranState(grid)
    if kind == "window":
        s["window"] = TransportWindow(ctx, case["nsteps"])
    if case["physics"]:
        s["turb"], s["moist"] = _physics(case, seed)
    return s


def run(s):
    case, ctx = s["case"], s["ctx"]
    kind = case["kind"]
    if kind in ("tracer", "gradient"):
        _put_all(ctx, "scalar", s["q"])
        ctx.scalar_transport_rk()
        _get_all(ctx, "scalar", s["q_out"])
        if kind == "tracer":
            return {"q": s["q_out"]}
        _put_all(ctx, "scalar_adj", s["lam"])
        ctx.scalar_transport_rk_adj()
        _get_all(ctx, "scalar_adj", s["lam_out"])
        return {"q": s["q_out"], "grad": s["lam_out"]}
    if kind == "diagnose":
        return {"mass": ctx.mass_sums(), "maxmin": ctx.tracer_maxmin(), "cfl": ctx.cfl_report().astype(np.float32)}
    if kind == "window":
        q0 = s["q"].clone().requires_grad_(True)
        qT = transport(q0, s["window"])
        qT.backward(s["lam"])
        return {"q": qT.detach(), "grad": q0.grad}
    if kind == "host":
        ctx.tend0()
        ctx.upload_state(s["up"], only=("thilt", "vmxet", "vmyet", "vmzet", "vmt"))
        ctx.prog_wrtv_rk()
        ctx.timeavg_momsc()
        for n, t in enumerate(s["sct"]):
            ctx.upload_scalar(n + 1, None, t)
        ctx.scalar_transport_rk()
        phys = ("thil", "rho", "press", "vxe", "vye", "vze", "wc")
        ctx.download_state(s["down"], only=phys)
        out = {n: s["down"].arrays[n] for n in phys}
        return {"state": out, "q": [ctx.download_scalar(n + 1) for n in range(case["ntr"])]}
    if case["physics"]:
        ctx.set_turbulence(*s["turb"])
        ctx.comp_alpha_press(*s["moist"])
    ctx.tend0()
    for _ in range(case["nacoust"]):
        ctx.prog_wrtv_rk()
    out = {}
    if kind == "longstep":
        ctx.timeavg_momsc()
        ctx.scalar_transport_rk()
        _get_all(ctx, "scalar", s["q_out"])
        out["q"] = s["q_out"]
        if case["adjoint"]:
            ctx.scalar_transport_rk_adj()
            _get_all(ctx, "scalar_adj", s["lam_out"])
            out["grad"] = s["lam_out"]
    for n, f in s["fields"].items():
        ctx.copy_field(n, 0, f.data_ptr(), 0)
    return dict(out, **s["fields"])


def work(case):
    """Inputs once and outputs once.  Dynamics per cell-level: 13 W fields, 4 W metrics (one
    FP64) and 6 V fields of 3 faces read, 9 W and 3 V fields written; a tracer step: vmasc
    (3 faces), wmasc, rho, rho_old and volti read, and each tracer (and adjoint) read and
    written.  Operations per cell-level and RK stage: about 500 for the dynamics, 110 per
    tracer and direction."""
    cells = (10 * case["nxp"] ** 2 + 2) * case["nlev"]
    e = 8 if case["prec"] == "f64" else 4
    kind, n = case["kind"], case["ntr"]
    dyn = {"bytes": e * (13 + 3 + 18 + 9 + 9) + 8 + (e + 12 if case["prec"] == "mixed" else 0), "flops": 3 * 500}
    tr = {"bytes": e * (7 + 2 * n), "flops": case["nrk_scal"] * 110 * n}
    b = f = 0.0
    if kind in ("acoustic", "longstep", "host", "window"):
        b, f = dyn["bytes"] * case["nacoust"], dyn["flops"] * case["nacoust"]
    if kind not in ("acoustic", "diagnose"):
        two = kind in ("gradient", "window") or case["adjoint"]
        b, f = b + tr["bytes"] * (2 if two else 1), f + tr["flops"] * (2 if two else 1)
    if kind == "host":
        b += 4 * 7 + 4 * (5 + 4) + 8 * n                       # the arrays that cross PCIe
    if kind == "diagnose":
        b, f = e * (7 + n) + 8, 4.0 * n + 20
    if kind == "window":                                       # forward, and again for the gradient
        b, f = b * case["nsteps"], f * case["nsteps"]
    return {"bytes": b * cells, "flops": f * cells}


# ------------------------------------------------------------------ the same passes in 64 bits
class _Tables:
    """The grid's tables as 64-bit device tensors; slot arrays are (N_W, 7) with the absent
    seventh (or sixth) slot pointing at the column itself with zero weights."""

    def __init__(self, g):
        a = g.arrays
        self.mza = g.mza
        npoly = torch.from_numpy(a["w_npoly"][1:]).to(DEV).long()
        on = torch.arange(7, device=DEV)[None, :] < npoly[:, None]
        own = torch.arange(g.mwa - 1, device=DEV)[:, None]
        self.slots = int(npoly.max())
        i = {n: torch.from_numpy(a[n][1:]).to(DEV).long() - 2 for n in ("w_iv", "w_iw", "v_iw", "v_im", "m_iv", "m_im")}
        self.nbr, self.face = torch.where(on, i["w_iw"], own), torch.where(on, i["w_iv"], 0)
        self.v_iw, self.v_im, self.m_iv, self.m_im = i["v_iw"], i["v_im"], i["m_iv"], i["m_im"]
        t = lambda n: torch.from_numpy(a[n][1:]).to(DEV).double()  # noqa: E731
        z = lambda n: torch.where(on, t(n)[:, :7], 0.0)  # noqa: E731
        self.dirv, self.gx, self.gy = z("w_dirv"), z("gxps_coef"), z("gyps_coef")
        self.ec = [z("w_ecvec_v" + x) for x in "xyz"]
        self.xxyy, self.xxyym = z("xx_yy"), t("xx_yy_m")
        side = (self.dirv > 0).long()                          # 0: this column is iw1, 1: iw2
        pair = lambda n: t(n)[self.face]  # noqa: E731                             (N_W, 7, 2)
        pick = lambda n, s: torch.where(on, pair(n).gather(2, s[:, :, None])[:, :, 0], 0.0)  # noqa: E731
        self.own = [pick(n, side) for n in ("v_dxps", "v_dyps", "xx0_v", "xy0_v", "yy0_v")]
        self.far = [pick(n, 1 - side) for n in ("v_dxps", "v_dyps", "xx0_v", "xy0_v", "yy0_v")]
        self.xyh = [torch.where(on, t("xy_h")[:, :, k], 0.0) for k in range(5)]
        self.volt = t("volt")
        self.volti = torch.where(self.volt > 0, 1.0 / self.volt, 0.0)
        lev = lambda n: torch.from_numpy(a[n]).to(DEV).double()  # noqa: E731
        self.lev = {n: lev(n) for n in ("dzim", "dzit", "zfacit", "zwgt_top8", "zwgt_bot8", "gdz_wgtm8", "gdz_wgtp8")}
        w = torch.from_numpy(a["a_w"]).to(DEV).double()        # [j, i, k]
        self.a11, self.a21, self.a12, self.a22 = w[0, 0], w[0, 1], w[1, 0], w[1, 1]
        self.t, self.g = t, g

    def grad(self, q, cx, cy):
        gx, gy = torch.zeros_like(q), torch.zeros_like(q)
        for j in range(self.slots):
            d = q[self.nbr[:, j]] - q
            gx = gx + cx[:, j, None] * d
            gy = gy + cy[:, j, None] * d
        return gx, gy

    def coefs(self, q, order):
        if order == 1:
            return []
        if order == 2:
            return list(self.grad(q, self.gx, self.gy))
        c = []
        for k in range(0, 5, 2):
            c += list(self.grad(q, self.xyh[k], self.xyh[min(k + 1, 4)]))
        return c[:5]

    def vertical(self, q, w):
        """The upwinded value at the top of each level (bounded quadratic)."""
        up = torch.cat([q[:, 1:], q[:, -1:]], 1)
        ds = up - q
        ds = torch.cat([torch.zeros_like(ds[:, :1]), ds[:, 1:-1], torch.zeros_like(ds[:, :1])], 1)
        dm = torch.cat([torch.zeros_like(ds[:, :1]), ds[:, :-1]], 1)
        bot, top = q + ds * self.a11 + dm * self.a21, q + ds * self.a12 + dm * self.a22
        u = torch.where(w < 0, torch.cat([bot[:, 1:], bot[:, -1:]], 1), top)
        return torch.cat([up[:, :1], u[:, 1:-1], q[:, -1:]], 1)


def _up(x):
    """The value one level below, zero below the lowest."""
    return torch.cat([torch.zeros_like(x[:, :1]), x[:, :-1]], 1)


def _dn(x):
    """The value one level above, the top's own at the top."""
    return torch.cat([x[:, 1:], x[:, -1:]], 1)


def _exact_tracer(T, q, vmasc, wmasc, rho, dt, order, nrk, sct=None):
    q0, x = q, q
    for frac in ((1 / 3, 0.5, 1.0) if nrk == 3 else (0.5, 1.0)):
        co = T.coefs(x, order)
        flux = torch.zeros_like(x)
        for j in range(T.slots):
            d, n = T.dirv[:, j, None], T.nbr[:, j]
            vm = vmasc[T.face[:, j]]
            fs, fn = x, x[n]
            for k, c in enumerate(co):
                fs = fs + T.own[k][:, j, None] * c
                fn = fn + T.far[k][:, j, None] * c[n]
            sel = torch.where(d < 0, vm < 0, ~(vm < 0))
            flux = flux + d * vm * (torch.where(sel, fn, fs) - q0)
        u = T.vertical(x, wmasc)
        flux = flux + _up(wmasc) * (_up(u) - q0) - wmasc * (u - q0)
        src = flux * T.volti if sct is None else flux * T.volti + sct
        x = q0 + frac * dt * src / rho
        x = torch.cat([x[:, 1:2], x[:, 1:]], 1)
    return x


def _exact_acoustic(T, case, S, tend=None):
    """One prog_wrtv_rk of the dry, order-2 dynamics with level-3 damping; S is updated."""
    p = _params(case)
    t, mza, dtm = T.t, T.mza, p.dtsm
    body = torch.zeros(mza, device=DEV, dtype=torch.float64)
    body[1:] = 1.0
    inner = body.clone()
    inner[-1] = 0.0
    arv, arw, volt, volti = t("arv"), t("arw"), T.volt, T.volti
    vsum = volt[T.v_iw[:, 0]] + volt[T.v_iw[:, 1]]
    volvi = torch.where(vsum > 0, 1.0 / vsum, 0.0)
    volwi = inner / torch.where(volt + _dn(volt) > 0, volt + _dn(volt), 1.0)
    del vsum
    iw1, iw2 = T.v_iw[:, 0], T.v_iw[:, 1]
    wn, vn = [t(n)[:, None] for n in ("wnx", "wny", "wnz")], [t(n)[:, None] for n in ("vnx", "vny", "vnz")]
    L = T.lev
    pwfac, pvfac = L["dzim"], t("dniv")[:, None] * L["zfacit"]
    rho0, rth0, wmc0, vmc0 = S["rho"], S["rho"] * S["thil"], S["wmc"], S["vmc"]
    ts = [0.0 if tend is None else tend[n] * volt for n in ("thilt", "vmxet", "vmyet", "vmzet")]
    # sixth-order divergence and vorticity damping of the horizontal wind
    div = torch.zeros_like(volt)
    for j in range(T.slots):
        div = div - T.dirv[:, j, None] * (arv * S["vmc"])[T.face[:, j]]
    div = div * volti
    for _ in range(2):
        d = torch.zeros_like(div)
        for j in range(T.slots):
            d = d + T.xxyy[:, j, None] * (div[T.nbr[:, j]] - div)
        div = d * body
    fd, fv = float(p.divh_damp_fact), float(p.vort_damp_fact)
    amin = torch.minimum(t("arw0")[iw1], t("arw0")[iw2])
    vmin = torch.minimum(volt[iw1], volt[iw2])
    vmt = (fd ** 3 / dtm * amin ** 2 * t("dniv"))[:, None] * (L["zfacit"] * L["dzit"] * body) * vmin * (div[iw2] - div[iw1])
    vort = torch.zeros((T.m_iv.shape[0], mza), device=DEV, dtype=torch.float64)
    im = torch.arange(T.m_iv.shape[0], device=DEV)
    for j in range(3):
        e = T.m_iv[:, j]
        sign = torch.where(T.v_im[e, 1] == im, 1.0, -1.0)
        vort = vort + (sign * t("dnv")[e] / t("arm0"))[:, None] * S["vc"][e] * body
    for _ in range(2):
        d = torch.zeros_like(vort)
        for j in range(3):
            d = d + T.xxyym[:, j, None] * (vort[T.m_im[:, j]] - vort)
        vort = d
    mmin = torch.minimum(t("arm0")[T.v_im[:, 0]], t("arm0")[T.v_im[:, 1]])
    fvor = (0.5 * t("dniu") / dtm * (-fv * mmin) ** 3)[:, None]
    vmt = vmt + fvor * (vort[T.v_im[:, 1]] - vort[T.v_im[:, 0]]) * (rho0[iw1] + rho0[iw2])
    del div, vort, vmin
    cpocv, rocv, fr = 1004.0 / 717.0, 287.0 / 717.0, 0.7
    pc = fr * cpocv
    for stage, frac in enumerate((1 / 3, 0.5, 1.0), start=1):
        dt = frac * dtm
        qs = [S["thil"], *S["ve"]]
        g = [T.grad(q, T.gx, T.gy) for q in qs]
        hflx, tt = torch.zeros_like(volt), [torch.zeros_like(volt) + x for x in ts]
        mca = S["vmc"] * arv
        for j in range(T.slots):
            d, n = T.dirv[:, j, None], T.nbr[:, j]
            vm = mca[T.face[:, j]]
            sel = torch.where(d < 0, vm < 0, ~(vm < 0))
            hflx = hflx + d * vm
            for k, q in enumerate(qs):
                fs = q + T.own[0][:, j, None] * g[k][0] + T.own[1][:, j, None] * g[k][1]
                fn = q[n] + T.far[0][:, j, None] * g[k][0][n] + T.far[1][:, j, None] * g[k][1][n]
                tt[k] = tt[k] + d * vm * torch.where(sel, fn, fs)
        del g
        rho = S["rho"]
        tt[1] = tt[1] + rho * volt * p.fcoriol * S["ve"][1]
        tt[2] = tt[2] - rho * volt * p.fcoriol * S["ve"][0]
        ups = [T.vertical(q, S["wmc"]) for q in qs]
        rth = rho * S["thil"]
        b10 = dt * volti
        b5 = S["alpha"] * rth.clamp(min=0.0) ** rocv * body
        dr, drt = b10 * hflx, b10 * tt[0]
        if stage > 1:
            dr, drt = dr + rho0 - rho, drt + rth0 - rth
        pex, rex = b5 * (rth + pc * drt), rho + fr * dr
        wm = wmc0 + dt * ((pex - _dn(pex)) * pwfac - (L["gdz_wgtm8"] * rex + L["gdz_wgtp8"] * _dn(rex)) +
                          sum(w * (x + _dn(x)) for w, x in zip(wn, tt[1:])) * volwi)
        b15, c8, c9 = b10 * b5, dt * pc, -dt * dt * fr
        b8, b7 = c8 * pwfac, dt * volwi
        b23, b24 = b8 * b15, b8 * _dn(b15)
        b25, b26 = c9 * volti * L["gdz_wgtm8"], c9 * _dn(volti) * L["gdz_wgtp8"]
        lo = -_up(arw) * (b7 * _up(S["wc"]) + b25 + b23 * _up(ups[0]))
        di = 1.0 + arw * (b25 - b26 + (b23 + b24) * ups[0])
        hi = _dn(arw) * (b7 * _dn(S["wc"]) + b26 - b24 * _dn(ups[0]))
        cp, dp = [None] * mza, [None] * mza                     # Thomas, levels 2..mza-1
        for k in range(1, mza - 1):
            den = di[:, k] - (lo[:, k] * cp[k - 1] if k > 1 else 0.0)
            cp[k] = hi[:, k] / den
            dp[k] = (wm[:, k] - (lo[:, k] * dp[k - 1] if k > 1 else 0.0)) / den
        w = torch.zeros_like(volt)
        for k in range(mza - 2, 0, -1):
            w[:, k] = dp[k] - (cp[k] * w[:, k + 1] if k < mza - 2 else 0.0)
        wma = w * arw * inner
        v = [wma * u for u in ups]
        rho_n = torch.where(body > 0, rho0 + dt * volti * (hflx + _up(wma) - wma), rho)
        drt = drt + b10 * (_up(v[0]) - v[0])
        press = torch.where(body > 0, b5 * (rth + pc * drt), S["press"])
        th = torch.where(body > 0, (rth + drt) / torch.where(rho_n != 0, rho_n, 1.0), S["thil"])
        tr = [x + _up(y) - y for x, y in zip(tt[1:], v[1:])]
        wden = L["zwgt_bot8"] * rho_n + L["zwgt_top8"] * _dn(rho_n)
        wc = torch.where(inner > 0, w / torch.where(wden != 0, wden, 1.0), S["wc"])
        wc = torch.cat([wc[:, 1:2], wc[:, 1:]], 1)
        S["thil"] = torch.cat([th[:, 1:2], th[:, 1:]], 1)
        S["rho"], S["press"], S["wc"] = rho_n, press, wc
        S["wmc"] = torch.where(inner > 0, w, S["wmc"])
        vm = vmc0 + dt * (vmt + (press[iw1] - press[iw2]) * pvfac +
                          sum(n * (x[iw1] + x[iw2]) for n, x in zip(vn, tr)) * volvi)
        S["vmc"] = torch.where(body > 0, vm, S["vmc"])
        vden = rho_n[iw1] + rho_n[iw2]
        S["vc"] = torch.where(body > 0, 2.0 * vm / torch.where(vden != 0, vden, 1.0), S["vc"])
        if stage == 2:
            S["vmasc"] = S["vmasc"] + vm * arv * body
        if stage == 3:
            S["wmasc"] = S["wmasc"] + wma
        wst = _up(wc) + wc
        ve = [0.5 * wst * n for n in wn]
        for j in range(T.slots):
            for k in range(3):
                ve[k] = ve[k] + T.ec[k][:, j, None] * S["vc"][T.face[:, j]]
        S["ve"] = [torch.cat([x[:, 1:2], x[:, 1:]], 1) for x in ve]


def exact(case, seed):
    kind = case["kind"]
    if kind == "window" or case["monot"] or case["mono_dyn"] or case["physics"]:
        return None
    if kind in ("acoustic", "longstep", "host") and case["order"] != 2:
        return None
    T = _Tables(_grid(case["nxp"], case["nlev"]))
    dev = lambda a: torch.from_numpy(a[1:]).to(DEV).double()  # noqa: E731
    out = {}
    q = _tracers(case, seed, _real(case)) if case["ntr"] else None
    dt, nacoust = _dt(case["nxp"]), case["nacoust"]
    sct = [None] * case["ntr"]
    if kind in ("tracer", "gradient", "diagnose"):
        w = _winds(case["nxp"], case["nlev"])
        vmasc, wmasc, rho = dev(w["vmasc"]), dev(w["wmasc"]), dev(w["rho"])
        if kind == "diagnose":
            rho = rho.to(torch.float64 if case["prec"] == "mixed" else _real(case)).double()
            lo, hi = q[:, :, 1:].amin((1, 2)), q[:, :, 1:].amax((1, 2))
            mass = (rho * T.volt)[:, 1:]
            sums = [mass.sum()] + [(mass * x[:, 1:].double()).sum() for x in q]
            return {"mass": torch.stack(sums).cpu(), "maxmin": torch.stack([hi, lo], 1).double().cpu(), "cfl": None}
    else:
        st = _jet(case["nxp"], case["nlev"]).arrays
        th, rho = _anomaly(case, seed)
        S = {n: dev(st[n]) for n in ("press", "wmc", "wc", "vmc", "vc")}
        S.update(thil=th, rho=rho, alpha=dev(st["alpha_press"]), ve=[dev(st[n]) for n in ("vxe", "vye", "vze")],
                 vmasc=torch.zeros_like(S["vmc"]), wmasc=torch.zeros_like(rho))
        tend = None
        if kind == "host":
            tend, sct = _tendencies(case, seed)
            tend, sct = {n: dev(a) for n, a in tend.items()}, [dev(a) for a in sct]
        if nacoust > 1:                # the damping keeps its last Laplacian between calls
            return None
        _exact_acoustic(T, case, S, tend)
        rho, vmasc, wmasc = S["rho"], S["vmasc"], S["wmasc"]
        if kind == "host":
            low = lambda x: torch.cat([torch.zeros_like(x[:1]), x], 0)  # noqa: E731   the dummy point
            out["state"] = {n: low(x) for n, x in (("thil", S["thil"]), ("rho", S["rho"]), ("press", S["press"]),
                                                   ("vxe", S["ve"][0]), ("vye", S["ve"][1]), ("vze", S["ve"][2]),
                                                   ("wc", S["wc"]))}
        else:
            out.update({n: S[n] for n in ("thil", "rho", "press", "wmc", "vmc")})
        del S
    if kind == "acoustic":
        return out
    rho = torch.where(rho != 0, rho, 1.0)
    two = kind == "gradient" or case["adjoint"]
    lam = _adjoints(case, seed, _real(case)) if two else None
    qs, gs = [], []
    for n in range(case["ntr"]):
        x = q[n].double().requires_grad_(two)
        y = _exact_tracer(T, x, vmasc, wmasc, rho, dt, case["order"], case["nrk_scal"], sct[n])
        if two:
            gs.append(torch.autograd.grad(y, x, lam[n].double())[0])
        qs.append(y.detach())
        del x, y
    if kind == "host":
        out["q"] = [torch.cat([torch.zeros_like(x[:1]), x], 0) for x in qs]
    else:
        out["q"] = torch.stack(qs)
    if two:
        out["grad"] = torch.stack(gs)
    return out
