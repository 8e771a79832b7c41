"""Tracer mass under steady winds with the two-ring stages, whose columns each sum their own
rounded weights: what leaves a cell and what enters its neighbours agree to rounding, not to
the bit.  Per step the mass after it (rho of its end) is compared with the mass before it (rho
of its start) in FP64 on the host, from the stored FP32 mixing ratios, and the differences are
added over the steps, so an error that the winds repeat every step adds up.

Bound: per step and cell about 9 roundings of half an ulp (u = 2**-24) of the cell's own mass
or less (the stored ratio and density, the flux sum's 40 terms at Courant numbers below 0.2),
3 u rms; independent between cells, so 3 u / sqrt(N) of the total with N = (sum m)^2 / sum m^2
the cells that carry the mass; the same in every step at worst; four times that: 12 K u /
sqrt(N).  One ulp of the same sign in every cell would exceed it at the first step."""

import numpy as np
import pytest

from olam_amd import abi
from olam_amd.gpu import Context
from helpers import tracer_case

pytestmark = pytest.mark.gpu

K, NTR = 20, 4


@pytest.mark.parametrize("nxp,nlev,prec,order,kernel", [
    (12, 16, "f32", 2, "k_tr_ring2"), (12, 70, "mixed", 2, "k_tr_ring2"), (12, 16, "f32", 3, "k_tr_ring2"),
    (21, 20, "f32", 2, "k_tr_ring2s"), (21, 20, "mixed", 3, "k_tr_ring2s"), (21, 70, "f32", 2, "k_tr_ring2s")])
def test_mass_under_steady_winds(grid_factory, nxp, nlev, prec, order, kernel):
    print(f"mass: NXP={nxp} L={nlev} {prec} order={order}", flush=True)
    grid = grid_factory(nxp, nlev)
    w, st, tr = tracer_case(grid, dt=300.0, ntr=NTR)
    rho = w["rho"] if prec == "mixed" else w["rho"].astype(np.float32).astype(np.float64)
    m0, m1 = ((r * grid.arrays["volt"])[1:, 1:] for r in (w["rho_old"].astype(np.float64), rho))
    g = Context(grid, abi.make_params(prec, num_scalar=NTR, dtsm=300.0, order=order), device=0)
    g.set_profiling(True)
    g.upload_state(st)
    for n in range(NTR):
        g.upload_scalar(n + 1, tr[n])
    q = [x[1:, 1:].astype(np.float64) for x in tr]
    total = [(m0 * x).sum() for x in q]
    cells = [t * t / ((m0 * x) ** 2).sum() for t, x in zip(total, q)]
    change = np.zeros(NTR)
    for _ in range(K):
        before = [(m0 * x).sum() for x in q]
        g.scalar_transport_rk(w["rho_old"])
        q = [g.download_scalar(n + 1)[1:, 1:].astype(np.float64) for n in range(NTR)]
        change += [((m1 * x).sum() - b) / t for x, b, t in zip(q, before, total)]
    assert g.kernel_profile()[kernel][0] == 3 * K
    g.close()
    for n in range(NTR):
        bound = 12 * K * 2.0 ** -24 / np.sqrt(cells[n])
        print(f"  tracer {n + 1}: {change[n]:.2e} of its mass in {K} steps, bound {bound:.2e}", flush=True)
        assert abs(change[n]) <= bound
