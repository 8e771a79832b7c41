"""The kernels that stage a block's rows in LDS against the oracle, on the smallest meshes
that take them and whose last block is partly filled: tracer stages and their adjoints from
4,096 columns on (NXP=21: 4,412, two tracers and more), the dynamics' flux sums from 8,192
one-wave columns on (NXP=29: 8,412); columns of 3, 63 and 64 levels, tall tracer columns, a
last group of one tracer, and monotone fluxes in the last stage only.

Tolerances, relative to the largest value: tracers as for the two-ring stage, FP32
3 * sqrt(40) * 2**-24 = 1.2e-6 taken as 2e-6, FP64 through FP32 downloads 1.2e-7; dynamics
exactly those of the gradient pass (the oracle's FP64 fields come down in FP32, so FP64 is
held to that comparison alone) and after two steps, a few FP32 ulps times the columns'
solve, 1e-5 of the oracle and 1e-4 for the vertical momentum, whose largest value is small.
"""

import numpy as np
import pytest

from olam_amd import abi, cases
from olam_amd.gpu import Context
from helpers import DYN_FIELDS, dyn_fields, rel_linf, tracer_case
from oracle import Oracle
from test_gpu_ring2 import TOL, _run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nlev,prec,order,ntr", [
    (3, "f32", 2, 2), (63, "f32", 2, 17), (24, "f64", 2, 3), (63, "mixed", 3, 3), (64, "f32", 2, 2), (70, "f64", 3, 2)])
def test_staged_tracers(grid_factory, nlev, prec, order, ntr):
    print(f"staged tracers: NXP=21 L={nlev} {prec} order={order} {ntr} tracers", flush=True)
    grid = grid_factory(21, nlev)
    w, st, tr = tracer_case(grid, dt=300.0, ntr=ntr)
    rng = np.random.default_rng(5)
    lam = [rng.standard_normal((grid.mwa, grid.mza)).astype(np.float32) for _ in range(ntr)]
    prm = abi.make_params(prec, num_scalar=ntr, dtsm=300.0, order=order)
    got = _run(Context(grid, prm, device=0), w, st, tr, lam)
    want = _run(Oracle(grid, prm), w, st, tr, lam)
    for n in range(ntr):
        e, ea = rel_linf(got[0][n], want[0][n]), rel_linf(got[1][n], want[1][n])
        print(f"  tracer {n + 1}: forward {e:.2e} adjoint {ea:.2e}")
        assert e <= TOL[prec] and ea <= TOL[prec]


@pytest.mark.parametrize("nlev,prec,mono", [
    (3, "f32", 0), (63, "f32", 0), (40, "mixed", 0), (30, "f64", 0), (20, "f32", 1), (64, "f32", 0)])
def test_staged_fluxes(grid_factory, nlev, prec, mono):
    print(f"staged fluxes: NXP=29 L={nlev} {prec} mono={mono}", flush=True)
    grid = grid_factory(29, nlev)
    jet = cases.jet_state(grid)
    prm = abi.make_params(prec, num_scalar=1, dtsm=300.0, ithil_monot=mono, iwind_monot=mono)
    # a run nudged by a zero density tendency takes the gradient pass: the same to the bit
    nudged = abi.make_params(prec, num_scalar=1, dtsm=300.0, ithil_monot=mono, iwind_monot=mono, nudflag=2,
                             nud_preserve_total_mass=0)
    f = []
    for be in (Context(grid, prm, device=0), Context(grid, nudged, device=0), Oracle(grid, prm)):
        be.upload_state(jet)
        be.tend0()
        be.prog_wrtv_rk()
        be.prog_wrtv_rk()
        f.append(dyn_fields(be, grid))
        be.close()
    for n in DYN_FIELDS:
        e = rel_linf(f[0][n], f[2][n])
        print(f"  {n:6s} {e:.2e}")
        assert np.array_equal(f[0][n], f[1][n])
        assert prec == "f64" or e < (1e-4 if n in ("wmc", "wc", "wmasc") else 1e-5)
