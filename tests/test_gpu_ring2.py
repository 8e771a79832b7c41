"""The two-ring tracer stage and its adjoint (csrc/kernels_ring2.h) against the oracle at
the sizes where they can go wrong: meshes whose rings meet around the sphere (NXP=1, 2) and
whose pentagons neighbour each other's rings (3), one-wave columns of 3 and 63 levels, tall
columns at the overlap of their two waves (64, 70), the tallest they take (123) and the
first they do not (124), one tracer and more than one group of them (17), a stage input
that differs at level 1, and tables whose slots are not cyclic, which take the gradient and
update passes instead.

Tolerances, relative to the largest value: FP32, three stages of about 40 rounded terms of
the size of the result or smaller, 3 * sqrt(40) * 2**-24 = 1.2e-6, taken as 2e-6 (the
adjoint of random weights has outputs a few times smaller than its terms); FP64 through
FP32 downloads, one FP32 rounding, 1.2e-7.  Implicit columns (wnoise=40, vertical Courant
numbers near 1000) run in FP64: there the FP32 oracle itself is 1e-4 to 1e-3 off the FP64
one, so it is no reference for FP32.
"""

import numpy as np
import pytest

from olam_amd import abi
from olam_amd.gpu import Context
from helpers import PermutedGrid, rel_linf, tracer_case
from oracle import Oracle

pytestmark = pytest.mark.gpu

TOL = {"f32": 2e-6, "mixed": 2e-6, "f64": 1.2e-7}


class ShuffledSlots(PermutedGrid):
    """The same grid with each W point's neighbour slots in a seeded random order."""

    def __init__(self, grid, seed=0):
        super().__init__(grid, seed)
        rng = np.random.default_rng(seed + 1)
        npoly = self.arrays["w_npoly"]
        order = np.tile(np.arange(7), (grid.mwa, 1))
        for i in range(1, grid.mwa):
            order[i, : npoly[i]] = rng.permutation(npoly[i])
        for k in ("w_iv", "w_iw", "w_im", "w_dirv", "w_ecvec_vx", "w_ecvec_vy", "w_ecvec_vz", "gxps_coef",
                  "gyps_coef", "xx_yy", "xy_h", "xy_hu"):
            a = self.arrays[k]
            ix = order if a.ndim == 2 else np.repeat(order[:, :, None], a.shape[2], 2)
            a[...] = np.take_along_axis(a, ix, 1)


def _run(be, w, st, tr, lam):
    be.upload_state(st)
    for n, q in enumerate(tr, start=1):
        be.upload_scalar(n, q)
        be.upload_scalar_adj(n, lam[n - 1])
    be.scalar_transport_rk(w["rho_old"])
    be.scalar_transport_rk_adj()
    out = ([be.download_scalar(n + 1) for n in range(len(tr))],
           [be.download_scalar_adj(n + 1) for n in range(len(tr))])
    be.close()
    return out


@pytest.mark.parametrize("nxp,nlev,prec,order,nrk,ntr,wnoise", [
    (1, 5, "f32", 2, 3, 2, 0.01), (2, 16, "f64", 2, 3, 3, 0.01), (3, 3, "f32", 2, 2, 1, 0.01),
    (6, 63, "f32", 2, 3, 17, 0.01), (6, 63, "f64", 3, 3, 3, 0.01), (5, 24, "mixed", 3, 2, 3, 0.01),
    (6, 24, "f64", 2, 3, 3, 40.0), (4, 64, "f32", 2, 3, 3, 0.01), (4, 70, "f64", 2, 3, 17, 0.01),
    (4, 70, "f64", 3, 3, 3, 40.0), (4, 123, "f32", 2, 3, 3, 0.01), (4, 124, "f32", 2, 3, 3, 0.01)])
def test_two_ring_stage(grid_factory, nxp, nlev, prec, order, nrk, ntr, wnoise):
    print(f"two rings: NXP={nxp} L={nlev} {prec} order={order} RK{nrk} {ntr} tracers wnoise={wnoise}", flush=True)
    grid = grid_factory(nxp, nlev)
    w, st, tr = tracer_case(grid, dt=300.0, ntr=ntr, wnoise=wnoise)
    rng = np.random.default_rng(5)
    tr[-1] = tr[-1].copy()
    tr[-1][:, 0] = 7.0                       # level 1 is not a copy of level 2
    lam = [rng.standard_normal((grid.mwa, grid.mza)).astype(np.float32) for _ in range(ntr)]
    prm = abi.make_params(prec, num_scalar=ntr, dtsm=300.0, order=order, nrk_scal=nrk)
    got = _run(Context(grid, prm, device=0), w, st, tr, lam)
    want = _run(Oracle(grid, prm), w, st, tr, lam)
    for n in range(ntr):
        e, ea = rel_linf(got[0][n], want[0][n]), rel_linf(got[1][n], want[1][n])
        print(f"  tracer {n + 1}: forward {e:.2e} adjoint {ea:.2e}")
        assert e <= TOL[prec] and ea <= TOL[prec]


@pytest.mark.parametrize("prec,order", [("f32", 2), ("f64", 3)])
def test_slots_in_any_order(grid_factory, prec, order):
    print(f"shuffled slots: NXP=6 L=20 {prec} order={order}", flush=True)
    grid = ShuffledSlots(grid_factory(6, 20), seed=3)
    w, st, tr = tracer_case(grid.base, dt=300.0, ntr=3)
    for n in ("vmasc",):
        st.arrays[n] = grid.fwd(st.arrays[n], "v")
    for n in ("wmasc", "rho"):
        st.arrays[n] = grid.fwd(st.arrays[n])
    w = dict(w, rho_old=grid.fwd(w["rho_old"]))
    tr = [grid.fwd(q) for q in tr]
    rng = np.random.default_rng(5)
    lam = [rng.standard_normal((grid.mwa, grid.mza)).astype(np.float32) for _ in range(3)]
    prm = abi.make_params(prec, num_scalar=3, dtsm=300.0, order=order)
    got = _run(Context(grid, prm, device=0), w, st, tr, lam)
    want = _run(Oracle(grid, prm), w, st, tr, lam)
    for n in range(3):
        e, ea = rel_linf(got[0][n], want[0][n]), rel_linf(got[1][n], want[1][n])
        print(f"  tracer {n + 1}: forward {e:.2e} adjoint {ea:.2e}")
        assert e <= TOL[prec] and ea <= TOL[prec]
