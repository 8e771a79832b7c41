// kernels_ring2.h -- explicit tracer stages and their adjoint as one pass over the
// two-ring stencil.
//
// With the winds given, an unlimited explicit stage is linear in the tracer, and its
// weights do not depend on which tracer it is.  The face value of update_scalar
// (scalar_transport_rk.F90:474-533) is the upwind cell's value plus its reconstruction
// terms (grad_t2d, grad_lib.f90:236-269, or grad_t2d_quadratic, :278-341) times the face
// offsets, and those terms are weighted sums of differences to that cell's neighbours, so
// the horizontal part of a column's update is
//     F = sum over the 18 cells r of its two rings of C_r (q_r - q_c) + (q_c - q0_c) S
// with C_r per level from the face mass fluxes and per-column constants of the mesh, and
// S the net inflow.  A wave forms the 18 weights of its column once and then spends 18
// gathers and 36 multiply-adds per tracer; no reconstruction terms are written to or read
// from memory, and order 3 costs what order 2 costs.  The adjoint is the transpose: the
// weights with which the 18 cells' updates read this column.
//
// Rings of a column with npoly 5 or 6 whose neighbours have 5 or 6 sides (numbering
// cyclic): ring 1 is n_0..n_5; ring 2 is mid_j (the other common neighbour of n_j and
// n_j+1) and far_j (beyond n_j, absent if n_j is a pentagon).  Absent cells point at the
// column itself with zero constants.  A mesh with any other neighbourhood keeps the
// gradient and update passes of kernels_tracer.h.
//
// What bounds it: the gathers, 19 rows of a column per tracer from L1 and L2 (4.9 KB,
// 14 TB/s at the size below), with 7 GB of compulsory HBM traffic per stage.  Measured at
// NXP=320, L=60, 10 tracers, FP32: forward stage 3.62 ms against 2.10 + 4.58 for
// k_tr_grad and k_tr_update, adjoint stage 4.51 against 5.25 + 3.26 for k_tr_adj01 and
// k_tr_adj2; NXP=48, L=60, 8 tracers, order 3: 0.075 against 0.108 + 0.261 and 0.083
// against 0.124 + 0.241; NXP=40, L=30, one FP64 tracer: 0.031 against 0.011 + 0.039.
// A cell that is not finite makes its two rings not finite (its weight may be zero).
#pragma once
#include "kernels_tracer.h"

// Mesh constants of the two-ring stencil (see ring2_tables in olamgpu.hip).
template <class R>
struct Ring2Tab {
  const int *cell;       // nw x 12: mid_0..mid_5, far_0..far_5
  const R *kf;           // nw x 36: per slot j {sum, prev, next, mid_j-1, mid_j, far_j}
  const int *face;       // nw x 24: faces n_j|n_j+1, n_j|mid_j-1, n_j|mid_j, n_j|far_j
  const unsigned *out;   // nw: bit i set where face i's positive flux leaves n_j
  const R *ka;           // nw x 42: per slot j {c, prev, next, mid_j-1, mid_j, far_j}, then own_j
};

// Rows of one tracer field read through a buffer resource: the lane's byte offset in a
// vector register, the column's in a scalar one, so a gather costs no address arithmetic.
// The host takes this path only where a field is smaller than 4 GiB.
template <class R>
struct Rows {
  __amdgpu_buffer_rsrc_t rs;
  __device__ __forceinline__ Rows(const R *p, unsigned bytes)
      : rs(__builtin_amdgcn_make_buffer_rsrc((void *)p, 0, (int)bytes, 0x00020000)) {}
  template <int AUX = 0>
  __device__ __forceinline__ R get(unsigned lane_bytes, unsigned col_bytes) const {
    if constexpr (sizeof(R) == 4) {
      return __builtin_bit_cast(R, __builtin_amdgcn_raw_buffer_load_b32(rs, (int)lane_bytes, (int)col_bytes, AUX));
    } else {
      return __builtin_bit_cast(R, __builtin_amdgcn_raw_buffer_load_b64(rs, (int)lane_bytes, (int)col_bytes, AUX));
    }
  }
};
constexpr int ROWS_NT = 2;   // non-temporal: rows read once

// Position of a wave: column, tracers and level.  A tall column's two waves overlap by
// four levels (the first holds levels 1..64 and stores 1..62, the second holds 61..124
// and stores from 63), so the vertical stencil, two levels each way, needs no exchange
// between them; columns of more than 124 levels keep the other passes.
constexpr int RING2_TALL_BASE = 60, RING2_TALL_MZA = RING2_TALL_BASE + WAVE;
struct RingItem { int c, n0, n1, l; bool own; };
template <bool TALL>
__device__ __forceinline__ RingItem ring_item(int nw, int ntr, int tpw) {
  const TrItem t = tr_item(nw, ntr, tpw, TALL ? 1 : 0);
  RingItem r;
  r.c = t.c; r.n0 = t.n0; r.n1 = t.n1;
  if constexpr (TALL) {
    const int lane = lane_id();
    const bool upper = t.l >= WAVE;
    r.l = upper ? RING2_TALL_BASE + lane : lane;
    r.own = upper ? lane >= 2 : lane < RING2_TALL_BASE + 2;
  } else {
    r.l = t.l;
    r.own = true;
  }
  return r;
}

template <class R, class RP, bool Q3, bool TALL>
__global__ __launch_bounds__(256) void k_tr_ring2(DMesh<R> m, Ring2Tab<R> t, TrStage<R, RP> a) {
  const RingItem ti = ring_item<TALL>(m.nw, a.ntr, a.tpw);
  const int c = ti.c;
  if (c >= m.nw) return;
  const int l = ti.l, k = l + 1, mza = m.mza;
  const unsigned ul = (unsigned)l;
  const bool act = k <= mza, body = act && k >= 2, inner = k >= 2 && k <= mza - 1;
  const long ldk = m.ldk, cb = (long)c * ldk;
  constexpr int NQ = Q3 ? 5 : 2;
  const R *off[5] = {m.w_dxs, m.w_dys, m.w_os[0][0], m.w_os[0][1], m.w_os[0][2]};
  const R *cof[5] = {Q3 ? m.w_q[0][0] : m.w_gxc, Q3 ? m.w_q[0][1] : m.w_gyc, m.w_q[0][2], m.w_q[0][3], m.w_q[0][4]};
  // weights: w_j is the inflow through face j, taken from n_j; the outflow carries this
  // column's own reconstruction, whose terms sum to b
  R w[6], b[NQ], S = R(0);
  unsigned row[18];
#pragma unroll
  for (int q = 0; q < NQ; ++q) b[q] = R(0);
#pragma unroll
  for (int j = 0; j < 6; ++j) {
    const int s = c * NSLOT + j;
    row[j] = (unsigned)m.w_nbr[s] * (unsigned)(ldk * sizeof(R));
    const R f = m.w_dirv[s] * ldl(a.vmasc + (long)m.w_face[s] * ldk, ul);
    w[j] = f > R(0) ? f : R(0);
    const R o = f - w[j];
    S = S + f;
#pragma unroll
    for (int q = 0; q < NQ; ++q) b[q] = b[q] + off[q][s] * o;
  }
#pragma unroll
  for (int i = 0; i < 12; ++i) row[6 + i] = (unsigned)t.cell[c * 12 + i] * (unsigned)(ldk * sizeof(R));
  R C[18];
  const R *kf = t.kf + (long)c * 36;
#pragma unroll
  for (int j = 0; j < 6; ++j) {
    const int jm = (j + 5) % 6, jp = (j + 1) % 6;
    R e = w[j];
#pragma unroll
    for (int q = 0; q < NQ; ++q) e = e + b[q] * cof[q][c * NSLOT + j];
    C[j] = e - w[j] * kf[6 * j] + w[jm] * kf[6 * jm + 2] + w[jp] * kf[6 * jp + 1];
    C[6 + j] = w[j] * kf[6 * j + 4] + w[jp] * kf[6 * jp + 3];
    C[12 + j] = w[j] * kf[6 * j + 5];
  }
  if (m.w_npoly[c] == 5) {        // n_4 and n_0 are neighbours; slot 5 reads the column itself
    C[0] = C[0] + w[4] * kf[6 * 4 + 2];
    C[4] = C[4] + w[0] * kf[1];
  }
  // vertical: with d(k) = q(k+1) - q(k) on levels 2..mza-1 the upwinded value at W level k
  // less q(k) is v0 d(k-1) + v1 d(k) + v2 d(k+1) (grad_z_quadratic, bounded)
  const R wm = ldl(a.wmasc + cb, ul);
  const R fexpl = R(1) - a.ffimp[(long)(a.istage - 1) * m.nw + c];
  const R wf = inner ? fexpl * wm : R(0);
  const int lp = min(l + 1, (int)ldk - 1);
  const bool neg = wm < R(0);
  const R v0 = neg ? R(0) : wf * m.aw22[l];
  const R v1 = neg ? wf * (R(1) + m.aw21[lp]) : wf * m.aw12[l];
  const R v2 = neg ? wf * m.aw11[lp] : R(0);
  S = S + fexpl * (shup(wm, 1) - wm);
  const R rf = (R)a.rho[cb + l];
  const R rinv = R(1) / (body ? rf : R(1));
  const R vt = ldl(m.volti + cb, ul);
  const unsigned fb = (unsigned)((size_t)m.nw * ldk * sizeof(R)), lb = ul * (unsigned)sizeof(R),
                 own = (unsigned)c * (unsigned)(ldk * sizeof(R));
  const bool start = a.q_in == a.q0;
  for (int n = ti.n0; n < ti.n1; ++n) {
    const long fo = n * a.tstride;
    const Rows<R> q(a.q_in + fo, fb);
    const R qc = q.get(lb, own);
    R qn[18];
#pragma unroll
    for (int i = 0; i < 18; ++i) qn[i] = q.get(lb, row[i]);
    const R q0 = start ? qc : Rows<R>(a.q0 + fo, fb).template get<ROWS_NT>(lb, own);
    const R st = a.sct ? Rows<R>(a.sct + fo, fb).template get<ROWS_NT>(lb, own) : R(0);
    R d = shdn(qc, 1) - qc;
    d = inner ? d : R(0);
    const R y = v0 * shup(d, 1) + v1 * d + v2 * shdn(d, 1);
    const R x = y - wf * d;                     // the same flux against the level above
    R F = (qc - q0) * S + (shup(x, 1) - y);
#pragma unroll
    for (int i = 0; i < 18; ++i) F = F + C[i] * (qn[i] - qc);
    R r = q0 + a.dtr * (st + vt * F) * rinv;
    const R lev1 = shdn(r, 1);                  // level 1 copies level 2
    if (k == 1) r = lev1;
    if (act && ti.own) st_nt(a.q_out + fo, cb + l, r);
  }
}

// volti / rho on the prognostic levels, zero elsewhere: what turns the adjoint of a stage
// output into that of the flux sum, shared by the stages of an adjoint step.
template <class R, class RP>
__global__ __launch_bounds__(256) void k_tr_vr(DMesh<R> m, const RP *rho, R *out) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (long)m.nw * m.ldk) return;
  const int k = (int)(i & (m.ldk - 1)) + 1;
  out[i] = (k >= 2 && k <= m.mza) ? m.volti[i] / (R)rho[i] : R(0);
}

// Transpose of k_tr_ring2: mu of the stage output to lq of the stage input and the scp0
// terms in lam0 (scheme as k_tr_adj01 and k_tr_adj2).  D_r is the weight with which the
// update of cell r reads this column: the face fluxes leaving this column and its ring-1
// cells m, through m's reconstruction coefficient that points back here.  Lane 0 carries
// level 2's weights, so what mu holds at level 1 (a copy of level 2 in the forward stage)
// is weighted as level 2 and then added there.
template <class R, class RP, bool Q3, bool TALL>
__global__ __launch_bounds__(256) void k_tr_ring2_adj(DMesh<R> m, Ring2Tab<R> t, TrAdj<R, RP> a, const R *vr) {
  const RingItem ti = ring_item<TALL>(m.nw, a.ntr, a.tpw);
  const int c = ti.c;
  if (c >= m.nw) return;
  const int l = ti.l, k = l + 1, mza = m.mza;
  const unsigned ul = (unsigned)l, um = ul ? ul : 1u;
  const bool act = k <= mza, body = act && k >= 2, inner = k >= 2 && k <= mza - 1;
  const long ldk = m.ldk, cb = (long)c * ldk;
  R D[18];
  unsigned row[18];
#pragma unroll
  for (int i = 0; i < 18; ++i) D[i] = R(0);
  const R *ka = t.ka + (long)c * 42;
  const int *f2 = t.face + (long)c * 24;
  const unsigned out = t.out[c];
  auto flux = [&](int i) {       // outflow of n_j positive
    const R v = ldl(a.vmasc + (long)f2[i] * ldk, um);
    return ((out >> i) & 1u) ? v : -v;
  };
  auto pos = [](R v) { return v > R(0) ? v : R(0); };
  R csum = R(0), rim[6], fix0 = R(0), fix4 = R(0);
#pragma unroll
  for (int j = 0; j < 6; ++j) rim[j] = flux(j);
#pragma unroll
  for (int j = 0; j < 6; ++j) {
    const int s = c * NSLOT + j, jm = (j + 5) % 6, jp = (j + 1) % 6;
    row[j] = (unsigned)m.w_nbr[s] * (unsigned)(ldk * sizeof(R));
    const R f = m.w_dirv[s] * ldl(a.vmasc + (long)m.w_face[s] * ldk, um);
    csum = csum + f;
    const R in = pos(f);
    R sum = ka[6 * j] * in;
    const R tp = ka[6 * j + 1] * pos(-rim[jm]), tn = ka[6 * j + 2] * pos(rim[j]);
    const R tmp_ = ka[6 * j + 3] * pos(flux(6 + j)), tmn = ka[6 * j + 4] * pos(flux(12 + j)),
            tf = ka[6 * j + 5] * pos(flux(18 + j));
    sum = sum + tp + tn + tmp_ + tmn + tf;
    D[j] = D[j] + ka[36 + j] * (in - f) - sum;
    D[jm] = D[jm] + tp;
    D[jp] = D[jp] + tn;
    if (j == 0) fix4 = tp;
    if (j == 4) fix0 = tn;
    D[6 + jm] = D[6 + jm] + tmp_;
    D[6 + j] = D[6 + j] + tmn;
    D[12 + j] = tf;
  }
  if (m.w_npoly[c] == 5) {        // n_4 and n_0 are neighbours, slot 5 is the column itself
    D[0] = D[0] + fix0;
    D[4] = D[4] + fix4;
    D[5] = R(0);
  }
#pragma unroll
  for (int i = 0; i < 12; ++i) row[6 + i] = (unsigned)t.cell[c * 12 + i] * (unsigned)(ldk * sizeof(R));
  R Dc = R(0);
  const unsigned fb = (unsigned)((size_t)m.nw * ldk * sizeof(R)), lb = ul * (unsigned)sizeof(R),
                 mb = um * (unsigned)sizeof(R), own = (unsigned)c * (unsigned)(ldk * sizeof(R));
  const Rows<R> gr(vr, fb);
#pragma unroll
  for (int i = 0; i < 18; ++i) {
    Dc = Dc - D[i];
    D[i] = D[i] * (a.dtr * gr.get(mb, row[i]));
  }
  const R g = a.dtr * gr.get(mb, own);
  Dc = Dc * g;
  // vertical transpose: upw(k) feeds F(k+1) with +wf and F(k) with -wf
  const R wm = ldl(a.wmasc + cb, ul);
  const R ff = a.ffimp[(long)(a.istage - 1) * m.nw + c];
  const R fexpl = R(1) - ff;
  const R cc = csum + fexpl * (shup(wm, 1) - wm);
  const R wf = inner ? fexpl * wm : R(0);
  const bool neg = wm < R(0);
  const bool neg_m1 = shup((int)neg, 1) != 0, neg_p1 = shdn((int)neg, 1) != 0;
  const int lp = min(l + 1, (int)ldk - 1);
  const R al = (inner && !neg) ? R(1) : R(0), be = (body && k >= 3 && neg_m1) ? R(1) : R(0);
  const R cm = (inner && k >= 3 && neg_m1) ? m.aw11[l] : R(0);
  const R c0 = inner ? (neg ? m.aw21[lp] : m.aw12[l]) : R(0);
  const R cp = (k >= 2 && k <= mza - 2 && !neg_p1) ? m.aw22[lp] : R(0);
  // on the first adjoint stage lam0 holds only what the implicit pass of this column wrote
  const bool rd0 = !a.first || ff > R(0.001);
  for (int n = ti.n0; n < ti.n1; ++n) {
    const long fo = n * a.tstride;
    const Rows<R> q(a.mu + fo, fb);
    const R mr = q.get(lb, own);
    R mn[18];
#pragma unroll
    for (int i = 0; i < 18; ++i) mn[i] = q.get(lb, row[i]);
    R l0 = rd0 ? Rows<R>(a.lam0 + fo, fb).template get<ROWS_NT>(lb, own) : R(0);
    const R below = shup(mr, 1);
    const R mu = k == 1 ? R(0) : (k == 2 ? mr + below : mr);
    const R nu = mu * g;
    if (body) l0 = l0 + mu - nu * cc;
    const R L = wf * (shdn(nu, 1) - nu);
    const R Lm = shup(L, 1);
    const R lds = cm * Lm + c0 * L + cp * shdn(L, 1);
    R acc = Dc * mr;
#pragma unroll
    for (int i = 0; i < 18; ++i) acc = acc + D[i] * mn[i];
    const R acc1 = shup(acc, 1);
    if (k == 2) acc = acc + acc1;
    R lq = acc + (al * L + be * Lm + (shup(lds, 1) - lds));
    if (!body) lq = R(0);
    if (a.last) lq = lq + l0;                   // stage 1 read q = scp0
    if (act && ti.own) {
      if (!a.last) st_nt(a.lam0 + fo, cb + l, l0);
      st_nt(a.lq + fo, cb + l, lq);
    }
  }
}
