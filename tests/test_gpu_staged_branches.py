"""The branches of the staged two-ring stages and their adjoints that need a mesh of 4,096
columns and more (NXP=21: 4,412): a tracer tendency, RK2 and RK3, implicit columns and a
limited final stage (with which the adjoint keeps its scp0 terms in an array instead of the
stages' mu), horizontal diffusion, one- and two-wave columns, the last block partly filled.
And which kernels run: each case names the launches it stands for, so that it fails where the
library falls back to others.

References: the same mesh with each column's slots shuffled, which the two-ring kernels do not
take, so the gradient and update passes run, compared at the working precision (copy_field)
over every level, and the oracle through FP32 downloads, level 1 too: after an explicit,
unlimited forward step it is a copy of level 2 and after an adjoint step zero, exactly.

Tolerances, relative to the largest value: the two sides each round about 40 terms of the
result's size per stage, 2 * 3 * sqrt(40) * eps / 2 = 19 eps, taken as 32 eps (adjoint outputs
are a few times smaller than their terms): 3.8e-6 in FP32, 7.1e-15 in FP64.  Columns solved
implicitly and limited stages amplify the difference of their inputs: 1e-11, as their parity
tests, and 1e-3 in FP32, as far as the FP32 oracle is from the FP64 one there.  Against the oracle in FP64 one FP32 rounding, 1.2e-7; in FP32 as the staged tracer
tests, 2e-6."""

import numpy as np
import pytest
import torch

from olam_amd import abi, cases
from olam_amd.gpu import Context
from helpers import DYN_FIELDS, dyn_fields, rel_linf, tracer_case
from oracle import Oracle
from test_gpu_ring2 import TOL, ShuffledSlots
from test_tracer_sgs_nudging import strong_turbulence

pytestmark = pytest.mark.gpu

EPS = {"f32": 2.0 ** -23, "mixed": 2.0 ** -23, "f64": 2.0 ** -52}
NTR = 3


def _full(g, name):
    """Every level of the tracers or their adjoints at the working precision."""
    dt = torch.float64 if g.params.precision == 2 else torch.float32
    out = torch.empty((NTR, g.grid.mwa - 1, g.grid.mza), dtype=dt, device="cuda")
    torch.cuda.synchronize()
    for n in range(NTR):
        g.copy_field(name, n + 1, out[n].data_ptr(), 0)
    torch.cuda.synchronize()
    return out.cpu().numpy()


def _step(be, w, st, tr, lam, sct, turb, what):
    be.upload_state(st)
    if turb is not None:
        be.set_turbulence(*turb)
        be.set_scalar_sgsmix(NTR, 0)
    for n in range(NTR):
        be.upload_scalar(n + 1, tr[n], sct if n == 1 else None)
        be.upload_scalar_adj(n + 1, lam[n])
    if what == "pdef":
        be.set_scalar_pdef(NTR, False)
    be.scalar_transport_rk(w["rho_old"])
    be.scalar_transport_rk_adj()


@pytest.mark.parametrize("nlev,prec,order,nrk,what", [
    (20, "f32", 2, 3, "sct"), (20, "f64", 2, 2, "sct"), (63, "f64", 2, 3, "sct"), (20, "f64", 3, 3, "sct"),
    (70, "f64", 2, 2, ""), (70, "f64", 2, 3, ""), (70, "f32", 3, 3, "sct"), (123, "f32", 2, 2, "sct"),
    (20, "f64", 2, 3, "implicit"), (70, "f64", 2, 2, "implicit"), (20, "f64", 3, 2, "implicit"),
    (20, "f64", 2, 3, "monot"), (20, "f64", 2, 3, "pdef"), (20, "f64", 3, 2, "pdef"), (70, "f64", 2, 3, "pdef"),
    (20, "f64", 2, 3, "sgs"), (70, "f64", 2, 2, "sgs")])
def test_staged_branches(grid_factory, nlev, prec, order, nrk, what):
    print(f"staged: NXP=21 L={nlev} {prec} order={order} RK{nrk} {what}", flush=True)
    grid = grid_factory(21, nlev)
    mono = {"monot": 1, "pdef": 2}.get(what, 0)
    w, st, tr = tracer_case(grid, dt=300.0, ntr=NTR, wnoise=40.0 if what == "implicit" else 0.01)
    st.arrays["rho"][:] = w["rho"]
    rng = np.random.default_rng(5)
    lam = [rng.standard_normal((grid.mwa, grid.mza)).astype(np.float32) for _ in range(NTR)]
    sct = None
    if what in ("sct", "pdef"):
        sct = np.zeros((grid.mwa, grid.mza), np.float32)
        sct[1:, 1:] = 1e-4 * tr[1][1:, 1:]
    turb = strong_turbulence(grid, st, 3) if what == "sgs" else None
    prm = abi.make_params(prec, num_scalar=NTR, dtsm=300.0, order=order, nrk_scal=nrk, iscal_monot=mono)

    g = Context(grid, prm, device=0)
    g.set_profiling(True)
    _step(g, w, st, tr, lam, sct, turb, what)
    ran = {k: v[0] for k, v in g.kernel_profile().items() if k.startswith("k_tr_")}
    staged = nrk - (1 if mono else 0)             # a limited final stage has its own passes
    # at 123 levels the rows of a block's widest rings are more than the adjoint's lanes carry
    adj = "k_tr_ring2_adj" if nlev == 123 else "k_tr_ring2s_adj"
    assert ran["k_tr_ring2s"] == staged and ran[adj] == staged, ran
    implicit = g.cfl_report()[3] > 0               # thin levels make some without wnoise=40
    assert implicit == (what == "implicit" or nlev == 123)
    assert ("k_tr_adj_implicit" in ran) == implicit and ("k_tr_adj_sct" in ran) == (what == "sgs"), ran
    assert ("k_tr_lim_adj1" in ran) == bool(mono) and ("k_tr_grad" in ran or "k_tr_grad3" in ran) == bool(mono), ran
    got = _full(g, "scalar"), _full(g, "scalar_adj")
    down = [g.download_scalar(n + 1) for n in range(NTR)], [g.download_scalar_adj(n + 1) for n in range(NTR)]
    g.close()
    if not mono and not implicit:                 # those passes leave level 1 as the stage before had it
        assert np.array_equal(got[0][:, :, 0], got[0][:, :, 1])
    assert not got[1][:, :, 0].any()

    o = Oracle(grid, prm)
    _step(o, w, st, tr, lam, sct, turb, what)
    tol = TOL[prec] if not implicit or prec == "f64" else 1e-3
    for n in range(NTR):
        ref = o.download_scalar(n + 1), o.download_scalar_adj(n + 1)
        e, ea = rel_linf(down[0][n], ref[0]), rel_linf(down[1][n], ref[1])
        e1 = float(np.abs(down[0][n][1:, 0].astype(np.float64) - ref[0][1:, 0]).max() / np.abs(ref[0][1:]).max())
        print(f"  oracle, tracer {n + 1}: forward {e:.2e}, level 1 {e1:.2e}, adjoint {ea:.2e}", flush=True)
        assert e <= tol and e1 <= tol and ea <= tol
    o.close()
    if mono:
        return                                    # scales where the correction vanishes are arbitrary

    s = ShuffledSlots(grid, seed=3)
    for n in ("wmasc", "rho"):
        st.arrays[n] = s.fwd(st.arrays[n])
    st.arrays["vmasc"] = s.fwd(st.arrays["vmasc"], "v")
    g = Context(s, prm, device=0)
    g.set_profiling(True)
    _step(g, {"rho_old": s.fwd(w["rho_old"])}, st, [s.fwd(q) for q in tr], [s.fwd(x) for x in lam],
          None if sct is None else s.fwd(sct), None if turb is None else tuple(s.fwd(x) for x in turb), what)
    ran = g.kernel_profile()
    assert "k_tr_update" in ran and not any("ring2" in k for k in ran), sorted(ran)
    ref = _full(g, "scalar")[:, s.pw], _full(g, "scalar_adj")[:, s.pw]
    g.close()
    tol = (1e-11 if prec == "f64" else 1e-3) if implicit else 32 * EPS[prec]
    for n in range(NTR):
        e = [float(np.abs(a[n] - b[n]).max() / np.abs(b[n]).max()) for a, b in zip(got, ref)]
        print(f"  gradient and update passes, tracer {n + 1}: forward {e[0]:.2e} adjoint {e[1]:.2e}", flush=True)
        assert max(e) <= tol


@pytest.mark.parametrize("nxp,nlev,prec,ntr,slots,fwd,adj", [
    (6, 20, "f32", 2, 0, "k_tr_ring2", "k_tr_ring2_adj"), (21, 20, "f32", 1, 0, "k_tr_ring2", "k_tr_ring2_adj"),
    (21, 20, "f32", 2, 0, "k_tr_ring2s", "k_tr_ring2s_adj"), (6, 123, "f64", 2, 0, "k_tr_ring2", "k_tr_ring2_adj"),
    (6, 124, "f32", 2, 0, "k_tr_update", "k_tr_adj01"), (6, 20, "f32", 2, 1, "k_tr_update", "k_tr_adj01")])
def test_tracer_kernels(grid_factory, nxp, nlev, prec, ntr, slots, fwd, adj):
    print(f"kernels: NXP={nxp} L={nlev} {prec} {ntr} tracers shuffled={slots}", flush=True)
    grid = grid_factory(nxp, nlev)
    g = Context(ShuffledSlots(grid) if slots else grid, abi.make_params(prec, num_scalar=ntr, dtsm=300.0), device=0)
    st = abi.FortranState(grid)
    st.arrays["rho"][:] = 1.0
    g.upload_state(st, only=("rho",))
    g.tend0()
    g.set_profiling(True)
    g.scalar_transport_rk()
    g.scalar_transport_rk_adj()
    ran = g.kernel_profile()
    g.close()
    for want, names in ((fwd, ("k_tr_ring2", "k_tr_ring2s", "k_tr_update")),
                        (adj, ("k_tr_ring2_adj", "k_tr_ring2s_adj", "k_tr_adj01"))):
        assert [x for x in names if x in ran] == [want] and ran[want][0] == 3, sorted(ran)


@pytest.mark.parametrize("nxp,nlev,prec,mono,nud,flux", [
    (29, 3, "f32", 0, 0, 3), (29, 63, "f32", 0, 0, 3), (29, 40, "mixed", 0, 0, 3), (29, 30, "f64", 0, 0, 3),
    (29, 63, "f64", 0, 0, 3), (29, 20, "f64", 1, 0, 2), (29, 64, "f64", 0, 0, 0), (28, 20, "f32", 0, 0, 0),
    (29, 20, "f64", 0, 1, 0)])
def test_flux_sums_run_and_match_the_oracle(grid_factory, nxp, nlev, prec, mono, nud, flux):
    """Stages that take k_dyn_flux, and two acoustic steps against the oracle: FP64 through
    FP32 downloads to one rounding."""
    print(f"flux sums: NXP={nxp} L={nlev} {prec} mono={mono} nudging={nud}", flush=True)
    grid = grid_factory(nxp, nlev)
    jet = cases.jet_state(grid)
    prm = abi.make_params(prec, num_scalar=1, dtsm=300.0, ithil_monot=mono, iwind_monot=mono,
                          nudflag=2 if nud else 0, nud_preserve_total_mass=0)
    f = []
    for be in (Context(grid, prm, device=0), Oracle(grid, prm)):
        be.upload_state(jet)
        be.tend0()
        if not f:
            be.set_profiling(True)
        be.prog_wrtv_rk()
        if not f:
            ran = {k: v[0] for k, v in be.kernel_profile().items()}
            assert ran.get("k_dyn_flux", 0) == flux and ran.get("k_dyn_grad", 0) == 3 - flux, ran
        be.prog_wrtv_rk()
        f.append({n: a.copy() for n, a in dyn_fields(be, grid).items()})
        be.close()
    for n in DYN_FIELDS:
        e = rel_linf(f[0][n], f[1][n])
        print(f"  {n:6s} {e:.2e}", flush=True)
        assert e <= (1.2e-7 if prec == "f64" else 1e-4 if n in ("wmc", "wc", "wmasc") else 1e-5)
