"""Mass sums and tracer extrema at the edges of their reductions (a mesh of 12 columns and
one with more columns than a pass of the grid takes, one and two waves per column, tracer
counts around the groups of 8) against numpy: the extrema exactly, the sums, of positive
terms in FP64, to 1e-13."""

import numpy as np
import pytest

from olam_amd import abi
from olam_amd.gpu import Context

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nxp,nlev,ntr,prec", [(1, 3, 1, "f32"), (3, 63, 8, "mixed"), (3, 64, 9, "f64"),
                                               (40, 12, 17, "f32"), (2, 70, 64, "f32")])
def test_sums_and_extrema(grid_factory, nxp, nlev, ntr, prec):
    print(f"sums: NXP={nxp} L={nlev} {ntr} tracers {prec}", flush=True)
    grid = grid_factory(nxp, nlev)
    rng = np.random.default_rng(ntr)
    shape = (grid.mwa, grid.mza)
    st = abi.FortranState(grid)
    st.arrays["rho"][:] = rng.uniform(0.1, 1.2, shape).astype(np.float32)
    g = Context(grid, abi.make_params(prec, num_scalar=ntr), device=0)
    g.upload_state(st, only=("rho",))
    q = [rng.lognormal(-20.0, 2.0, shape).astype(np.float32) for _ in range(ntr)]
    q[0][:, 0] = np.nan                      # level 1 is not prognostic
    q[-1][:, 1:] *= -1.0
    if grid.mza > 4:
        q[0][1, 3] = np.nan                  # skipped by the extrema; its sum is not a number
    for n in range(ntr):
        g.upload_scalar(n + 1, q[n])
    mm, mass = g.tracer_maxmin(), g.mass_sums()
    g.close()
    m = st.arrays["rho"][1:, 1:] * grid.arrays["volt"][1:, 1:]
    assert abs(mass[0] - m.sum()) <= 1e-13 * m.sum()
    for n in range(ntr):
        x = q[n][1:, 1:]
        assert mm[n, 0] == np.nanmax(x) and mm[n, 1] == np.nanmin(x), n
        want = (m * x.astype(np.float64)).sum()
        assert np.isnan(want) and np.isnan(mass[1 + n]) or abs(mass[1 + n] - want) <= 1e-13 * abs(want), n
