"""A mass flux or a density that is not finite in a tracer step and its adjoint: the points
that are not finite afterwards are the oracle's, the others hold its values within the
two-ring tests' tolerance.  A face flux that is a NaN counts as positive (it is not below
zero) and takes its value from the first of its columns, in the adjoint too."""

import numpy as np
import pytest

from olam_amd import abi
from olam_amd.gpu import Context
from helpers import tracer_case
from oracle import Oracle
from test_gpu_ring2 import TOL, _run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("what", ["vmasc", "rho", "wmasc"])
@pytest.mark.parametrize("nxp,nlev,prec,order,nrk", [
    (12, 16, "f32", 2, 2), (12, 16, "f64", 3, 2), (12, 70, "mixed", 2, 2), (21, 20, "f32", 2, 2),
    (21, 20, "f64", 2, 3), (21, 70, "f32", 2, 2)])
def test_nonfinite_fluxes(grid_factory, nxp, nlev, prec, order, nrk, what):
    print(f"not finite {what}: NXP={nxp} L={nlev} {prec} order={order} RK{nrk}", flush=True)
    grid = grid_factory(nxp, nlev)
    mza, nw, nv = grid.mza, grid.mwa - 1, grid.mva - 1
    w, st, tr = tracer_case(grid, dt=300.0, ntr=2, wnoise=0.0)
    rng = np.random.default_rng(9)
    lam = [rng.standard_normal((grid.mwa, mza)).astype(np.float32) for _ in tr]
    a = st.arrays[what]
    penta = int(np.flatnonzero(grid.arrays["w_npoly"][1:] == 5)[3]) + 1
    if what == "vmasc":
        at = [1 + nv // 3, int(grid.arrays["w_iv"][penta, 1]) - 1]
    else:
        at = [1 + nw // 3, penta]
    for i, v, l in zip(at, (np.nan, np.nan), (mza // 2, min(mza - 3, 60))):
        a[i, l] = v
    prm = abi.make_params(prec, num_scalar=2, dtsm=300.0, order=order, nrk_scal=nrk)
    got = _run(Context(grid, prm, device=0), w, st, tr, lam)
    with np.errstate(invalid="ignore"):
        want = _run(Oracle(grid, prm), w, st, tr, lam)
    for d, name in enumerate(("forward", "adjoint")):
        for n in range(2):
            g, o = got[d][n][1:, 1:].astype(np.float64), want[d][n][1:, 1:].astype(np.float64)
            fg, fo = np.isfinite(g), np.isfinite(o)
            both = fg & fo
            err = np.abs(g[both] - o[both]).max() / np.abs(o[both]).max()
            print(f"  {name} {n + 1}: not finite {(~fg).sum()} oracle {(~fo).sum()} differ {(fg != fo).sum()} "
                  f"others {err:.2e}", flush=True)
            assert (~fo).any() and np.array_equal(fg, fo)
            assert err <= TOL[prec]


def test_any_face(grid_factory):
    """Each face of a small mesh in turn: none is read with a weight of zero by columns that
    have no such face."""
    print("not finite vmasc: every face of NXP=4", flush=True)
    grid = grid_factory(4, 5)
    w, st, tr = tracer_case(grid, dt=300.0, ntr=1, wnoise=0.0)
    lam = np.random.default_rng(9).standard_normal((grid.mwa, grid.mza)).astype(np.float32)
    prm = abi.make_params("f32", num_scalar=1, dtsm=300.0, nrk_scal=2)
    backends = Context(grid, prm, device=0), Oracle(grid, prm)
    flux = st.arrays["vmasc"]
    for e in range(1, grid.mva):
        keep, flux[e, 3] = flux[e, 3], np.nan
        out = []
        for be in backends:
            be.upload_state(st)
            be.upload_scalar(1, tr[0])
            be.upload_scalar_adj(1, lam)
            be.scalar_transport_rk(w["rho_old"])
            be.scalar_transport_rk_adj()
            out.append([np.isfinite(a[1:, 1:]) for a in (be.download_scalar(1), be.download_scalar_adj(1))])
        flux[e, 3] = keep
        assert (~out[1][0]).any() and (~out[1][1]).any()
        assert np.array_equal(out[0][0], out[1][0]), e
        assert np.array_equal(out[0][1], out[1][1]), e
    for be in backends:
        be.close()
