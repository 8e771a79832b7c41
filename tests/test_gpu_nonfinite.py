"""Where a NaN or an infinity in a tracer (or in an adjoint) goes in one tracer step: to the
columns and levels that the face values and the vertical reconstruction of the upwind side
carry it to, as in the oracle, and no further.  The points that are not finite afterwards are
the oracle's, exactly; the others hold the oracle's values within the two-ring tests'
tolerance.  Gathered and staged stages, one- and two-wave columns, orders 2 and 3, a pentagon,
its neighbours, the lowest and the highest level, the overlap of a tall column's waves, and
levels without wind (there a face of no flow is taken from one side all the same)."""

import numpy as np
import pytest

from olam_amd import abi
from olam_amd.gpu import Context
from helpers import tracer_case
from oracle import Oracle
from test_gpu_ring2 import TOL, _run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nxp,nlev,prec,order,nrk,still", [
    (12, 16, "f32", 2, 3, 0), (12, 16, "f64", 3, 2, 0), (12, 70, "mixed", 2, 3, 0), (12, 16, "f32", 2, 2, 1),
    (21, 20, "f32", 2, 3, 0), (21, 20, "f64", 2, 2, 0), (21, 20, "f32", 3, 3, 0), (21, 70, "f32", 2, 2, 0),
    (21, 20, "f32", 2, 2, 1)])
def test_nonfinite_stays_upwind(grid_factory, nxp, nlev, prec, order, nrk, still):
    print(f"not finite: NXP={nxp} L={nlev} {prec} order={order} RK{nrk} still={still}", flush=True)
    grid = grid_factory(nxp, nlev)
    mza, nw = grid.mza, grid.mwa - 1
    w, st, tr = tracer_case(grid, dt=300.0, ntr=4)
    rng = np.random.default_rng(9)
    if still:                                # no wind, of either sign, in the lower half
        for name in ("vmasc", "wmasc"):
            a = st.arrays[name]
            a[:, : mza // 2 + 2] = np.where(rng.random((a.shape[0], mza // 2 + 2)) < 0.5, 0.0, -0.0)
    lam = [rng.standard_normal((grid.mwa, mza)).astype(np.float32) for _ in tr]
    penta = int(np.flatnonzero(grid.arrays["w_npoly"][1:] == 5)[3]) + 1
    beside = int(grid.arrays["w_iw"][penta, 0]) - 1
    levels = [1, mza // 2, mza - 1, min(mza - 2, 61)]                # 2, the middle, mza, a tall wave's seam
    cells = [penta, beside, 1 + nw // 3, 1 + (2 * nw) // 3]
    for f in (tr, lam):
        for n, v in enumerate((np.nan, np.inf, -np.inf, np.nan)):
            f[n] = f[n].copy()
            f[n][cells[n], levels[n]] = v
            f[n][cells[n - 1], levels[n - 2]] = v
    prm = abi.make_params(prec, num_scalar=4, dtsm=300.0, order=order, nrk_scal=nrk)
    got = _run(Context(grid, prm, device=0), w, st, tr, lam)
    with np.errstate(invalid="ignore"):
        want = _run(Oracle(grid, prm), w, st, tr, lam)
    for d, name in enumerate(("forward", "adjoint")):
        for n in range(4):
            g, o = got[d][n][1:, 1:].astype(np.float64), want[d][n][1:, 1:].astype(np.float64)
            fg, fo = np.isfinite(g), np.isfinite(o)
            err = np.abs(g - o)[fg & fo].max() / np.abs(o[fg & fo]).max()
            print(f"  {name} {n + 1}: not finite {(~fg).sum()} oracle {(~fo).sum()} differ {(fg != fo).sum()} "
                  f"others {err:.2e}", flush=True)
            assert (~fo).any() and np.array_equal(fg, fo)
            assert err <= TOL[prec]
