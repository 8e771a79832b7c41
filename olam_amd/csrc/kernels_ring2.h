// kernels_ring2.h -- explicit tracer stages and their adjoint as one pass over the
// two-ring stencil, and the dynamics' flux sums from the same staged rows.
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
// Two forms.  k_tr_ring2 and k_tr_ring2_adj gather the 19 rows of a column per tracer; the
// requests from L1 to L2 bound them (0.6 of the rows miss L1).  k_tr_ring2s and
// k_tr_ring2s_adj stage the rows of 16 (12) consecutive columns in LDS, 4 rows a column,
// and run at the memory's rate per tracer plus the weights once per wave (about 240 and
// 400 vector instructions).  Measured per stage, forward and adjoint, staged / gathered /
// as gradient and update passes (k_tr_grad + k_tr_update, k_tr_adj01 + k_tr_adj2):
// NXP=160, L=60, 10 tracers, FP32: 0.66 / 0.93 / 1.69 and 0.83 / 1.15 / 2.15 ms;
// NXP=64, L=70, 20 tracers: 0.33 / 0.63 / 1.04 and 0.39 / 0.73 / 1.31 ms;
// NXP=48, L=60, 8 tracers, order 3: 0.056 / 0.071 / 0.368 and 0.067 / 0.084 / 0.365 ms.
// Over 40 steps of 8 FP32 tracers on 40,962 columns, <L q, lam> and <q, L^T lam> differ by
// 2.1e-7 |q||lam| / sqrt(N) rms (4.9e-7 for the gradient and update passes).
// Zero weights and values that are not finite: 0 times such a value is not zero, so a sum over
// all 18 cells would carry a NaN to both rings whatever the wind.  Where a sum comes out not
// finite, it is formed again in those lanes without the cells and levels that the upwind side
// does not read (skip), and the values that are not finite are those of the gradient and
// update passes, for tracers, adjoints, densities and fluxes.  Where all is finite that costs one
// comparison a tracer and some 5 % more instructions for the weights, which the weights held as
// formed (formed) give back.  Without / with it, forward and adjoint, us: NXP=160, L=60, 10
// tracers 658 / 662 and 835 / 827; NXP=64, L=70, 20 tracers 327 / 329 and 410 / 388; one FP64
// tracer at NXP=60, L=60 58.9 / 58.6 and 86.5 / 87.8; 8 FP32 tracers at NXP=16, L=60 14.9 / 15.6
// and 16.2 / 16.7.  Reading the fluxes again where it happens, instead of keeping skip, was slower
// (gradient of 4 tracers at NXP=160 3.64 -> 3.90 ms).
#pragma once
#include "kernels_tracer.h"

// Record of one column: its indices and constants, each in one run of memory.  A wave
// reads it with one vector load per 64 words, lane i the word i, and broadcasts words with
// readlane as it needs them; read with scalar loads, a few registers at a time, the record
// alone cost a wave several memory latencies (0.43 of 0.77 ms at 256,002 columns).
enum {
  R2_NBR = 0, R2_CELL = 6, R2_FACE = 18,   // n_j; mid_j, far_j; faces of the column
  R2_OUTER = 24,                           // faces n_j|n_j+1, n_j|mid_j-1, n_j|mid_j, n_j|far_j
  R2_OUT = 48,                             // bit i set where outer face i's positive flux leaves n_j
  R2_NPOLY = 49,
  R2_PLACE = 50, R2_PLACEA = 55,           // places of the 18 cells and the column among its block's rows, bytes
  R2_GRAD = 60,                            // places of n_0..n_5 and the column among the block's gradients, bytes
  R2_INTS = 62,
  // forward constants: dirv, then off and cof (nq terms x 6), then kf, per slot j {sum, prev,
  // next, mid_j-1, mid_j, far_j}
  R2_DIRV = 0, R2_OFF = 6,
  // adjoint constants: dirv, then ka, per slot j {c, prev, next, mid_j-1, mid_j, far_j}, then own_j
  R2_KA = 6, R2_KOWN = 42, R2_NKA = 48
};
__host__ __device__ constexpr int r2_cof(int nq) { return R2_OFF + 6 * nq; }
__host__ __device__ constexpr int r2_kf(int nq) { return R2_OFF + 12 * nq; }
__host__ __device__ constexpr int r2_nkf(int nq) { return R2_OFF + 12 * nq + 36; }
template <class R>
struct Ring2Tab {
  const int *ints;       // nw x R2_INTS
  const R *kf, *ka;      // nw x r2_nkf, nw x R2_NKA
};
__device__ __forceinline__ float lane_word(float v, int i) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), i));
}
__device__ __forceinline__ double lane_word(double v, int i) {
  const long long w = __builtin_bit_cast(long long, v);
  const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)w, i),
                 hi = (unsigned)__builtin_amdgcn_readlane((int)(w >> 32), i);
  return __builtin_bit_cast(double, (long long)(((unsigned long long)hi << 32) | lo));
}
struct RecI {
  int v;
  __device__ __forceinline__ explicit RecI(const int *t, int c) {
    const int lane = lane_id();
    v = lane < R2_INTS ? t[(long)c * R2_INTS + lane] : 0;
  }
  __device__ __forceinline__ int operator[](int i) const { return __builtin_amdgcn_readlane(v, i); }
};
template <class R, int N>
struct RecK {
  static constexpr int NV = (N + WAVE - 1) / WAVE;
  R v[NV];
  __device__ __forceinline__ RecK(const R *t, int c) {
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int x = i * WAVE + lane_id();
      v[i] = x < N ? t[(long)c * N + x] : R(0);
    }
  }
  __device__ __forceinline__ R operator[](int i) const { return lane_word(v[i / WAVE], i % WAVE); }
};

// The word with the sign bit.
__device__ __forceinline__ unsigned sign_word(float v) { return __builtin_bit_cast(unsigned, v); }
__device__ __forceinline__ unsigned sign_word(double v) { return (unsigned)(__builtin_bit_cast(unsigned long long, v) >> 32); }

// v, and infinity for a NaN: a mass flux that is a NaN is not below zero, so its face takes the
// value of the positive flux's side and must not count as one without flow.
__device__ __forceinline__ float nan_up(float v) { return fminf(v, __builtin_inff()); }
__device__ __forceinline__ double nan_up(double v) { return fmin(v, __builtin_inf()); }

// shdn(v, 1) and shup(v, 1) with zero in the lane that has no source, in the form that the
// compiler folds into the instruction using it.
template <int CTRL>
__device__ __forceinline__ float dpp0(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, true));
}
template <int CTRL>
__device__ __forceinline__ double dpp0(double v) {
  const long long w = __builtin_bit_cast(long long, v);
  const unsigned lo = (unsigned)__builtin_amdgcn_update_dpp(0, (int)w, CTRL, 0xF, 0xF, true),
                 hi = (unsigned)__builtin_amdgcn_update_dpp(0, (int)(w >> 32), CTRL, 0xF, 0xF, true);
  return __builtin_bit_cast(double, (long long)(((unsigned long long)hi << 32) | lo));
}
template <class R> __device__ __forceinline__ R above0(R v) { return dpp0<0x130>(v); }
template <class R> __device__ __forceinline__ R below0(R v) { return dpp0<0x138>(v); }

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

template <class R>
__device__ __forceinline__ unsigned field_bytes(const DMesh<R> &m) {
  return (unsigned)((size_t)m.nw * m.ldk * sizeof(R));
}

// Position of a wave: column, tracers and level.  A tall column's two waves overlap by
// four levels (the first holds levels 1..64 and stores 1..62, the second holds 61..124
// and stores from 63), so the vertical stencil, two levels each way, needs no exchange
// between them; columns of more than 124 levels keep the other passes.  blockIdx.y is the
// tracer group, so every wave of a block runs the same number of tracers.  Waves past the
// last column repeat it and store nothing.
constexpr int RING2_TALL_BASE = 60, RING2_TALL_MZA = RING2_TALL_BASE + WAVE;
struct RingItem { int b, c, n0, n1, l; bool own; };
template <bool TALL, int NW>
__device__ __forceinline__ RingItem ring_item(int nw, int ntr, int tpw) {
  RingItem r;
  r.b = xcd_block(blockIdx.x, gridDim.x);
  const int w = __builtin_amdgcn_readfirstlane(r.b * NW + (threadIdx.x >> 6));
  const int lane = lane_id();
  r.n0 = blockIdx.y * tpw;
  r.n1 = min(ntr, r.n0 + tpw);
  r.c = TALL ? w >> 1 : w;
  r.l = lane;
  r.own = r.c < nw;
  if constexpr (TALL) {
    const bool upper = w & 1;
    if (upper) r.l = RING2_TALL_BASE + lane;
    r.own = r.own && (upper ? lane >= 2 : lane < RING2_TALL_BASE + 2);
  }
  r.c = min(r.c, nw - 1);
  return r;
}

// Staging of a tracer's rows in LDS.  The 16 consecutive columns of a forward block (8
// tall ones) have about 64 cells in their rings (45) where their waves would gather 19 rows
// each: the block reads every row once, 16 bytes a lane, one tracer ahead of the one it
// computes from the other of two buffers, one barrier per tracer.  A row keeps the levels
// in use only, so what lies above them in a lane's read is the next row's.
constexpr int RING2_NWF = 16, RING2_NWA = 12;      // waves of a staged block, forward and adjoint
struct Ring2Stage {
  const int *count;      // per block: rows staged
  const int *cells;      // blocks x nmax: their columns
  int nmax;
  unsigned pitch, magic; // bytes of a row (a multiple of 16), 2^32 / pitch rounded up
  unsigned bytes;        // of one buffer
};
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
template <class R, int NCH, int NW>
struct Stager {
  unsigned to, from[NCH];
  bool get_[NCH];
  u32x4 v[NCH];
  __device__ __forceinline__ Stager(const Ring2Stage &t, int b, int ldk) {
    const unsigned total = (unsigned)t.count[b] * t.pitch;
    to = threadIdx.x * 16u;
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
      const unsigned at = to + (unsigned)(i * NW) * 1024u, cell = __umulhi(at, t.magic);
      get_[i] = at < total;
      from[i] = get_[i] ? (unsigned)t.cells[b * t.nmax + (int)cell] * (unsigned)(ldk * sizeof(R)) + (at - cell * t.pitch)
                        : 0u;
      v[i] = u32x4{0u, 0u, 0u, 0u};
    }
  }
  __device__ __forceinline__ void get(const Rows<R> &q) {
#pragma unroll
    for (int i = 0; i < NCH; ++i)
      if (get_[i]) v[i] = __builtin_amdgcn_raw_buffer_load_b128(q.rs, (int)from[i], 0, 0);
  }
  __device__ __forceinline__ void put(unsigned char *buf) const {
#pragma unroll
    for (int i = 0; i < NCH; ++i)
      if (get_[i]) *reinterpret_cast<u32x4 *>(buf + to + (unsigned)(i * NW) * 1024u) = v[i];
  }
};
template <class R>
__device__ __forceinline__ R lds_row(const unsigned char *buf, unsigned off) {
  return *reinterpret_cast<const R *>(buf + off);
}

// The first N weights as formed: the compiler does not form them, or parts of them, again where
// they are used, which spills scalar registers (k_tr_ring2 in FP64 40, none with it).
template <int N, class R>
__device__ __forceinline__ void formed(R *w) {
#pragma unroll
  for (int i = 0; i < N; ++i) asm volatile("" : "+v"(w[i]));
}

// Weights of one column for the forward stage (see the head of this file), and what the
// vertical part and the update need of the column.
template <class R>
struct RingFwd {
  R C[18], S, v0, v1, v2, wf, vt, rinv;
  unsigned skip;         // bit j: n_j is not upwind of face j; bit 6: the flux at this W level is not down
};
template <class R, class RP, bool Q3>
__device__ __forceinline__ void ring_fwd(const DMesh<R> &m, const RecI &I, const RecK<R, r2_nkf(Q3 ? 5 : 2)> &K,
                                         const TrStage<R, RP> &a, int c, int l, RingFwd<R> &f) {
  const int k = l + 1, mza = m.mza;
  const bool body = k <= mza && k >= 2, inner = k >= 2 && k <= mza - 1;
  const long ldk = m.ldk, cb = (long)c * ldk;
  const unsigned rowb = (unsigned)(ldk * sizeof(R)), fb = field_bytes(m), lb = (unsigned)l * (unsigned)sizeof(R),
                 own = (unsigned)c * rowb;
  const Rows<R> vr(a.vmasc, (unsigned)m.nv * rowb);
  constexpr int NQ = Q3 ? 5 : 2;
  constexpr int KF = r2_kf(NQ), COF = r2_cof(NQ);
  // w_j is the inflow through face j, taken from n_j; the outflow carries this column's
  // own reconstruction, whose terms sum to b
  R w[6], b[NQ], S = R(0);
#pragma unroll
  for (int q = 0; q < NQ; ++q) b[q] = R(0);
  R vm[6];
#pragma unroll
  for (int j = 0; j < 6; ++j) vm[j] = vr.get(lb, (unsigned)I[R2_FACE + j] * rowb);
  const R wm = Rows<R>(a.wmasc, fb).get(lb, own);
  const R rf = (R)a.rho[cb + l];
  f.vt = Rows<R>(m.volti, fb).get(lb, own);
#pragma unroll
  for (int j = 0; j < 6; ++j) {
    const R x = K[R2_DIRV + j] * (vm[j] + R(0));        // -0 only where a face without flow is taken from here
    f.skip = (j ? f.skip : 0u) | ((sign_word(x) >> (31 - j)) & (1u << j));
    w[j] = x > R(0) ? x : R(0);
    const R o = x - w[j];
    S = S + x;
#pragma unroll
    for (int q = 0; q < NQ; ++q) b[q] = b[q] + K[R2_OFF + 6 * q + j] * o;
  }
#pragma unroll
  for (int j = 0; j < 6; ++j) {
    const int jm = (j + 5) % 6, jp = (j + 1) % 6;
    R e = w[j];
#pragma unroll
    for (int q = 0; q < NQ; ++q) e = e + b[q] * K[COF + 6 * q + j];
    f.C[j] = e - w[j] * K[KF + 6 * j] + w[jm] * K[KF + 6 * jm + 2] + w[jp] * K[KF + 6 * jp + 1];
    f.C[6 + j] = w[j] * K[KF + 6 * j + 4] + w[jp] * K[KF + 6 * jp + 3];
    f.C[12 + j] = w[j] * K[KF + 6 * j + 5];
  }
  if (I[R2_NPOLY] == 5) {         // n_4 and n_0 are neighbours; slot 5 reads the column itself
    f.skip |= 1u << 5;
    f.C[0] = f.C[0] + w[4] * K[KF + 6 * 4 + 2];
    f.C[4] = f.C[4] + w[0] * K[KF + 1];
  }
  formed<18>(f.C);
  // vertical: with d(k) = q(k+1) - q(k) on levels 2..mza-1 the upwinded value at W level k
  // less q(k) is v0 d(k-1) + v1 d(k) + v2 d(k+1) (grad_z_quadratic, bounded)
  const R fexpl = R(1) - a.ffimp[(long)(a.istage - 1) * m.nw + c];
  f.wf = inner ? fexpl * wm : R(0);
  const int lp = min(l + 1, (int)ldk - 1);
  const bool neg = wm < R(0);
  f.skip |= neg ? 0u : 64u;
  f.v0 = neg ? R(0) : f.wf * m.aw22[l];
  f.v1 = neg ? f.wf * (R(1) + m.aw21[lp]) : f.wf * m.aw12[l];
  f.v2 = neg ? f.wf * m.aw11[lp] : R(0);
  f.S = S + fexpl * (below0(wm) - wm);
  f.rinv = R(1) / (body ? rf : R(1));
}
// Keeps the rarely run second sum from sharing masks, addresses and loads with the first and
// from loading ahead, which would hold registers throughout: v is new to the compiler, and
// known only after `after`.
template <class R>
__device__ __forceinline__ void opaque(unsigned &v, R &after) {
  asm volatile("" : "+v"(v), "+v"(after));
}
// The flux sum from the column's value, scp0 and the 18 cells' values; qn(i, 0) is called once
// per cell.  GATED: only what the upwind side reads.
template <bool GATED, class R, class F>
__device__ __forceinline__ R ring_fwd_sum(const RingFwd<R> &f, R qc, R q0, bool inner, F &&qn) {
  unsigned skip = f.skip, zero = 0u;
  if constexpr (GATED) opaque(skip, qc);
  auto unless = [&](unsigned bits, R v) { return GATED && (skip & bits) == bits ? R(0) : v; };
  R d = above0(qc) - qc;
  d = inner ? d : R(0);
  const R da = unless(64u, above0(d)), dm = below0(d);      // moves with every lane, then chosen
  const R db = GATED && !(skip & 64u) ? R(0) : dm;
  const R y = f.v0 * db + f.v1 * d + f.v2 * da;
  const R x = y - f.wf * d;                     // the same flux against the level above
  R F0 = (qc - q0) * f.S + (below0(x) - y), F1 = R(0);
  // ring 1 is always read: by the neighbour's own value or by this column's reconstruction
  auto cells = [](int i) { return i < 6 ? ~0u : (1u << (i % 6)) | (i < 12 ? 1u << ((i + 1) % 6) : 0u); };
#pragma unroll
  for (int i = 0; i < 18; i += 2) {
    if constexpr (GATED) opaque(zero, F0);
    F0 = F0 + f.C[i] * unless(cells(i), qn(i, zero) - qc);
    F1 = F1 + f.C[i + 1] * unless(cells(i + 1), qn(i + 1, zero) - qc);
  }
  return F0 + F1;
}
// true where a wave has to form its sum again
template <class R>
__device__ __forceinline__ bool any_not_finite(R v, bool where) {
  return __builtin_expect(__ballot(where && !__builtin_isfinite(v)) != 0, 0);
}
// The new value from the column's value, scp0, tendency and the 18 cells' values.
template <class R, class F>
__device__ __forceinline__ R ring_fwd_value(const RingFwd<R> &f, R qc, R q0, R st, R dtr, bool inner, bool body, int k,
                                            F &&qn) {
  R F0 = ring_fwd_sum<false>(f, qc, q0, inner, qn);
  if (any_not_finite(F0, body)) {
    const R g = ring_fwd_sum<true>(f, qc, q0, inner, qn);
    F0 = __builtin_isfinite(F0) ? F0 : g;
  }
  R r = q0 + dtr * (st + f.vt * F0) * f.rinv;
  const R lev1 = above0(r);                     // level 1 copies level 2
  return k == 1 ? lev1 : r;
}

template <class R, class RP, bool Q3, bool TALL>
__global__ __launch_bounds__(256) void k_tr_ring2(DMesh<R> m, Ring2Tab<R> t, TrStage<R, RP> a) {
  const RingItem ti = ring_item<TALL, WPB>(m.nw, a.ntr, a.tpw);
  const int c = ti.c, l = ti.l, k = l + 1, mza = m.mza;
  const bool inner = k >= 2 && k <= mza - 1, body = k >= 2 && k <= mza;
  const long cb = (long)c * m.ldk;
  const unsigned rowb = (unsigned)(m.ldk * sizeof(R)), fb = field_bytes(m), lb = (unsigned)l * (unsigned)sizeof(R),
                 own = (unsigned)c * rowb;
  const RecI I(t.ints, c);
  const RecK<R, r2_nkf(Q3 ? 5 : 2)> K(t.kf, c);
  RingFwd<R> f;
  ring_fwd<R, RP, Q3>(m, I, K, a, c, l, f);
  unsigned row[18];
#pragma unroll
  for (int i = 0; i < 18; ++i) row[i] = (unsigned)I[R2_NBR + i] * rowb;
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
    const R r = ring_fwd_value(f, qc, q0, st, a.dtr, inner, body, k, [&](int i, unsigned) { return qn[i]; });
    if (k <= mza && ti.own) st_nt(a.q_out + fo, cb + l, r);
  }
}

template <class R, class RP, bool Q3, bool TALL, int NCH>
__global__ __launch_bounds__(RING2_NWF * WAVE, sizeof(R) == 4 ? 8 : 1) void k_tr_ring2s(DMesh<R> m, Ring2Tab<R> t, Ring2Stage sg,
                                                               TrStage<R, RP> a) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const RingItem ti = ring_item<TALL, RING2_NWF>(m.nw, a.ntr, a.tpw);
  const int c = ti.c, l = ti.l, k = l + 1, mza = m.mza;
  const bool inner = k >= 2 && k <= mza - 1, body = k >= 2 && k <= mza;
  const long cb = (long)c * m.ldk;
  const unsigned rowb = (unsigned)(m.ldk * sizeof(R)), fb = field_bytes(m), lb = (unsigned)l * (unsigned)sizeof(R),
                 own = (unsigned)c * rowb;
  const RecI I(t.ints, c);
  const RecK<R, r2_nkf(Q3 ? 5 : 2)> K(t.kf, c);
  Stager<R, NCH, RING2_NWF> st_(sg, ti.b, m.ldk);
  const bool start = a.q_in == a.q0;
  R q0n = R(0), stn = R(0);
  auto fetch = [&](int n) {
    const long fo = n * a.tstride;
    st_.get(Rows<R>(a.q_in + fo, fb));
    if (!start) q0n = Rows<R>(a.q0 + fo, fb).template get<ROWS_NT>(lb, own);
    if (a.sct) stn = Rows<R>(a.sct + fo, fb).template get<ROWS_NT>(lb, own);
  };
  fetch(ti.n0);
  RingFwd<R> f;
  ring_fwd<R, RP, Q3>(m, I, K, a, c, l, f);
  unsigned row[19];
#pragma unroll
  for (int i = 0; i < 19; ++i) row[i] = (((unsigned)I[R2_PLACE + i / 4] >> (8 * (i % 4))) & 255u) * sg.pitch;
  st_.put(smem_raw);
  __syncthreads();
  for (int n = ti.n0; n < ti.n1; ++n) {
    const unsigned char *buf = smem_raw + ((n - ti.n0) & 1) * sg.bytes + lb;
    const R qc = lds_row<R>(buf, row[18]);
    const R q0 = start ? qc : q0n, st = stn;
    const bool more = n + 1 < ti.n1;
    if (more) fetch(n + 1);
    const R r = ring_fwd_value(f, qc, q0, st, a.dtr, inner, body, k,
                               [&](int i, unsigned z) { return lds_row<R>(buf, row[i] + z); });
    if (k <= mza && ti.own) st_nt(a.q_out + n * a.tstride, cb + l, r);
    if (more) {
      st_.put(smem_raw + ((n + 1 - ti.n0) & 1) * sg.bytes);
      __syncthreads();
    }
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
//
// With no implicit column and no limited stage (on) the scp0 terms need no array of their
// own: the buffers of the earlier stages' mu are still there, and the last stage adds
// mu_s - nu_s cc of every stage s to lq, smallest first, so the result is rounded once at
// its own size instead of once per stage.
template <class R>
struct AdjHist {
  int on;
  const R *mu3, *mu2;    // mu of the final stage (the adjoint at entry) and, in RK3, of stage 2
  R dt3, dt2;            // their time steps
};
template <class R>
struct RingAdj {
  R D[18], Dc, g, gc, cc, wf, al, be, cm, c0, cp;
  unsigned skip;         // bit i: cell 6 + i is not read; bits 12, 13: the levels below (cm) and above (cp)
  bool rd0;
};
// vr(i): volti / rho of cell i (18: this column) at the lane's weight level.
// FORMED weights are held as formed (formed()): all, or those that leave k_tr_ring2_adj in FP64
// its 4 waves per SIMD (12: 117 registers; 18: 135 and 3 waves; 60 levels, one tracer, order 2 at
// NXP=60 87.6 us, 103 with 18 of them spilled to 128 registers).  0, the FP32 k_tr_ring2s_adj,
// which a branch suits better (NXP=160, L=60, 10 tracers 827 us, 845 with 18; NXP=64, L=70, 20
// tracers 388 and 411): one that sets the weights of cells that are not read to zero where a
// density is not finite, as the gated sum does with their products.
template <int FORMED, class R, class RP, class F>
__device__ __forceinline__ void ring_adj(const DMesh<R> &m, const RecI &I, const RecK<R, R2_NKA> &K,
                                         const TrAdj<R, RP> &a, int c, int l, RingAdj<R> &f, F &&vr) {
  const int k = l + 1, mza = m.mza;
  const bool body = k <= mza && k >= 2, inner = k >= 2 && k <= mza - 1;
  const long ldk = m.ldk;
  const unsigned rowb = (unsigned)(ldk * sizeof(R)), lb = (unsigned)l * (unsigned)sizeof(R),
                 mb = (l ? (unsigned)l : 1u) * (unsigned)sizeof(R);
  const Rows<R> vf(a.vmasc, (unsigned)m.nv * rowb);
  R *D = f.D;
#pragma unroll
  for (int i = 0; i < 18; ++i) D[i] = R(0);
  // every flux first, then the weights
  R vm[6], vo[24];
#pragma unroll
  for (int j = 0; j < 6; ++j) vm[j] = vf.get(mb, (unsigned)I[R2_FACE + j] * rowb);
#pragma unroll
  for (int i = 0; i < 24; ++i) vo[i] = vf.get(mb, (unsigned)I[R2_OUTER + i] * rowb);
  const unsigned out = (unsigned)I[R2_OUT];
#pragma unroll
  for (int i = 0; i < 24; ++i)                  // outflow of n_j positive, -0 only where n_j does not give a face without flow its value
    vo[i] = nan_up(vo[i] + R(0)) * (((out >> i) & 1u) ? R(1) : R(-1));
  const R wm = Rows<R>(a.wmasc, field_bytes(m)).get(lb, (unsigned)c * rowb);
  auto pos = [](R v) { return v > R(0) ? v : R(0); };
  R csum = R(0), fix0 = R(0), fix4 = R(0);
  unsigned skip0 = 0u, skip1 = 0xfc0u;          // no flow from n_j to mid_j and far_j; from n_j+1 to mid_j
#pragma unroll
  for (int j = 0; j < 6; ++j) {
    const int jm = (j + 5) % 6, jp = (j + 1) % 6;
    const R x = K[R2_DIRV + j] * vm[j];
    csum = csum + x;
    const R in = pos(x);
    R sum = K[R2_KA + 6 * j] * in;
    const R tp = K[R2_KA + 6 * j + 1] * pos(-vo[jm]), tn = K[R2_KA + 6 * j + 2] * pos(vo[j]);
    const R tmp_ = K[R2_KA + 6 * j + 3] * pos(vo[6 + j]), tmn = K[R2_KA + 6 * j + 4] * pos(vo[12 + j]),
            tf = K[R2_KA + 6 * j + 5] * pos(vo[18 + j]);
    sum = sum + tp + tn + tmp_ + tmn + tf;
    D[j] = D[j] + K[R2_KOWN + j] * (in - x) - sum;
    D[jm] = D[jm] + tp;
    D[jp] = D[jp] + tn;
    if (j == 0) fix4 = tp;
    if (j == 4) fix0 = tn;
    D[6 + jm] = D[6 + jm] + tmp_;
    D[6 + j] = D[6 + j] + tmn;
    D[12 + j] = tf;
    skip0 |= ((sign_word(vo[12 + j]) >> (31 - j)) & (1u << j)) | ((sign_word(vo[18 + j]) >> (25 - j)) & (64u << j));
    skip1 |= (sign_word(vo[6 + j]) >> (31 - jm)) & (1u << jm);
  }
  if (I[R2_NPOLY] == 5) {         // n_4 and n_0 are neighbours, slot 5 is the column itself
    skip0 |= 1u << 5;
    skip1 |= 1u << 4;
    D[0] = D[0] + fix0;
    D[4] = D[4] + fix4;
    D[5] = R(0);
  }
  f.skip = skip0 & skip1;
  // the weights of a column sum to zero; its own is summed ring by ring from the smallest
  // terms on (far, mid, ring 1), not one rounding after another at the size of the sum
  auto six = [&](int b) { return ((D[b] + D[b + 3]) + (D[b + 1] + D[b + 4])) + (D[b + 2] + D[b + 5]); };
  const R Dc = -((six(12) + six(6)) + six(0));
#pragma unroll
  for (int i = 0; i < 18; ++i) D[i] = D[i] * vr(i);
  if constexpr (FORMED > 0) {
    formed<FORMED>(D);
  } else if (any_not_finite((six(12) + six(6)), true)) {
#pragma unroll
    for (int i = 0; i < 12; ++i) D[6 + i] = (f.skip >> i) & 1u ? R(0) : D[6 + i];
  }
  const R gc = vr(18);
  f.gc = body ? gc : R(0);
  f.g = a.dtr * f.gc;
  f.Dc = Dc * gc;
  // vertical transpose: upw(k) feeds F(k+1) with +wf and F(k) with -wf
  const R ff = a.ffimp[(long)(a.istage - 1) * m.nw + c];
  const R fexpl = R(1) - ff;
  f.cc = csum + fexpl * (below0(wm) - wm);
  f.wf = inner ? fexpl * wm : R(0);
  const bool neg = wm < R(0);
  const bool neg_m1 = shup((int)neg, 1) != 0, neg_p1 = shdn((int)neg, 1) != 0;
  const int lp = min(l + 1, (int)ldk - 1);
  f.al = (inner && !neg) ? R(1) : R(0);
  f.be = (body && k >= 3 && neg_m1) ? R(1) : R(0);
  const bool below = inner && k >= 3 && neg_m1, above = k >= 2 && k <= mza - 2 && !neg_p1;
  f.skip |= (below ? 0u : 1u << 12) | (above ? 0u : 1u << 13);
  f.cm = below ? m.aw11[l] : R(0);
  f.c0 = inner ? (neg ? m.aw21[lp] : m.aw12[l]) : R(0);
  f.cp = above ? m.aw22[lp] : R(0);
  // on the first adjoint stage lam0 holds only what the implicit pass of this column wrote
  f.rd0 = !a.first || ff > R(0.001);
}
// what mu holds at level 1 counts as level 2's
template <class R>
__device__ __forceinline__ R ring_fold(R mr, bool body, int k) {
  const R below = below0(mr);
  return body ? (k == 2 ? mr + below : mr) : R(0);
}
// lq from the column's mu (mr as read, nu of the stage) and its cells'; GATED as in
// ring_fwd_sum
template <bool GATED, class R, class F>
__device__ __forceinline__ R ring_adj_sum(const RingAdj<R> &f, R mr, R nu, R dtr, int k, F &&mn) {
  unsigned skip = f.skip, zero = 0u;
  if constexpr (GATED) opaque(skip, nu);
  auto unless = [&](unsigned bit, R v) { return GATED && (skip & bit) ? R(0) : v; };
  const R L = f.wf * (above0(nu) - nu);
  const R Lm = below0(L);
  const R lds = f.cm * unless(1u << 12, Lm) + f.c0 * L + f.cp * unless(1u << 13, above0(L));
  R acc = f.Dc * mr, acb = R(0);
#pragma unroll
  for (int i = 0; i < 18; i += 2) {
    if constexpr (GATED) opaque(zero, acc);
    // the product: a cell that is not read has no weight, whatever its density
    acc = acc + (i < 6 ? f.D[i] * mn(i, zero) : unless(1u << (i - 6), f.D[i] * mn(i, zero)));
    acb = acb + (i < 6 ? f.D[i + 1] * mn(i + 1, zero) : unless(1u << (i - 5), f.D[i + 1] * mn(i + 1, zero)));
  }
  acc = acc + acb;
  const R acc1 = below0(acc);
  if (k == 2) acc = acc + acc1;
  return dtr * acc + (f.al * L + f.be * Lm + (below0(lds) - lds));
}
// lq, and the stage's scp0 terms
template <class R, class F>
__device__ __forceinline__ R ring_adj_value(const RingAdj<R> &f, R mr, R &mu, R &nucc, R dtr, bool body, int k,
                                            F &&mn) {
  mu = ring_fold(mr, body, k);
  const R nu = mu * f.g;
  nucc = nu * f.cc;
  R lq = ring_adj_sum<false>(f, mr, nu, dtr, k, mn);
  if (any_not_finite(lq, body)) {
    const R g = ring_adj_sum<true>(f, mr, nu, dtr, k, mn);
    lq = __builtin_isfinite(lq) ? lq : g;
  }
  return body ? lq : R(0);
}

// The own-column rows a stage reads besides mu: lam0, or at the last stage of an AdjHist
// the earlier stages' mu.  The stage writes over one of them, so a lane reads only what it
// stores itself: not the levels that the other wave of a tall column stores, and nothing in a
// wave past the last column.
template <class R, class RP>
__device__ __forceinline__ void ring_adj_rows(const TrAdj<R, RP> &a, const AdjHist<R> &h, bool rd0, const R *&p1,
                                              const R *&p2) {
  p1 = h.on ? (a.last ? h.mu3 : nullptr) : (rd0 ? a.lam0 : nullptr);
  p2 = h.on && a.last ? h.mu2 : nullptr;
}
template <class R, class RP>
__device__ __forceinline__ void ring_adj_store(const TrAdj<R, RP> &a, const AdjHist<R> &h, const RingAdj<R> &f, R lq,
                                               R mu, R nucc, R p, R q, bool body, int k, bool st, int n, long i) {
  const long fo = n * a.tstride;
  R r = lq;
  if (h.on) {
    if (a.last) {               // stage 1 read q = scp0
      const R mu3 = ring_fold(p, body, k), mu2 = ring_fold(q, body, k);
      const R s = (lq + (mu - nucc)) + (mu2 - f.cc * (f.gc * (h.dt2 * mu2 + h.dt3 * mu3)));
      r = body ? mu3 + s : R(0);
    }
  } else {
    const R l0 = body ? p + mu - nucc : p;
    if (a.last) r = lq + l0;
    else if (st) st_nt(a.lam0 + fo, i, l0);
  }
  if (st) st_nt(a.lq + fo, i, r);
}

template <class R, class RP, bool TALL>
__global__ __launch_bounds__(256) void k_tr_ring2_adj(DMesh<R> m, Ring2Tab<R> t, TrAdj<R, RP> a, AdjHist<R> h,
                                                      const R *vr) {
  const RingItem ti = ring_item<TALL, WPB>(m.nw, a.ntr, a.tpw);
  const int c = ti.c, l = ti.l, k = l + 1, mza = m.mza;
  const bool act = k <= mza, body = act && k >= 2;
  const long cb = (long)c * m.ldk;
  const unsigned rowb = (unsigned)(m.ldk * sizeof(R)), fb = field_bytes(m), lb = (unsigned)l * (unsigned)sizeof(R),
                 mb = (l ? (unsigned)l : 1u) * (unsigned)sizeof(R);
  const RecI I(t.ints, c);
  const RecK<R, R2_NKA> K(t.ka, c);
  unsigned row[19];
#pragma unroll
  for (int i = 0; i < 18; ++i) row[i] = (unsigned)I[R2_NBR + i] * rowb;
  row[18] = (unsigned)c * rowb;
  const Rows<R> gr(vr, fb);
  RingAdj<R> f;
  ring_adj<sizeof(R) == 4 ? 18 : 12>(m, I, K, a, c, l, f, [&](int i) { return gr.get(mb, row[i]); });
  const R *p1, *p2;
  ring_adj_rows(a, h, f.rd0, p1, p2);
  for (int n = ti.n0; n < ti.n1; ++n) {
    const long fo = n * a.tstride;
    const Rows<R> q(a.mu + fo, fb);
    const R mr = q.get(lb, row[18]);
    R mn[18];
#pragma unroll
    for (int i = 0; i < 18; ++i) mn[i] = q.get(lb, row[i]);
    R p = R(0), q2 = R(0);
    if (p1 && ti.own) p = Rows<R>(p1 + fo, fb).template get<ROWS_NT>(lb, row[18]);
    if (p2 && ti.own) q2 = Rows<R>(p2 + fo, fb).template get<ROWS_NT>(lb, row[18]);
    R mu, nucc;
    const R lq = ring_adj_value(f, mr, mu, nucc, a.dtr, body, k, [&](int i, unsigned) { return mn[i]; });
    ring_adj_store(a, h, f, lq, mu, nucc, p, q2, body, k, act && ti.own, n, cb + l);
  }
}

template <class R, class RP, bool TALL, int NCH>
__global__ __launch_bounds__(RING2_NWA * WAVE, sizeof(R) == 4 ? 6 : 1) void k_tr_ring2s_adj(DMesh<R> m, Ring2Tab<R> t, Ring2Stage sg,
                                                                   TrAdj<R, RP> a, AdjHist<R> h, const R *vr) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const RingItem ti = ring_item<TALL, RING2_NWA>(m.nw, a.ntr, a.tpw);
  const int c = ti.c, l = ti.l, k = l + 1, mza = m.mza;
  const bool act = k <= mza, body = act && k >= 2;
  const long cb = (long)c * m.ldk;
  const unsigned rowb = (unsigned)(m.ldk * sizeof(R)), fb = field_bytes(m), lb = (unsigned)l * (unsigned)sizeof(R),
                 mb = (l ? (unsigned)l : 1u) * (unsigned)sizeof(R), own = (unsigned)c * rowb;
  const RecI I(t.ints, c);
  const RecK<R, R2_NKA> K(t.ka, c);
  Stager<R, NCH, RING2_NWA> st_(sg, ti.b, m.ldk);
  const bool rd0 = !a.first || a.ffimp[(long)(a.istage - 1) * m.nw + c] > R(0.001);
  const R *p1, *p2;
  ring_adj_rows(a, h, rd0, p1, p2);
  R pn = R(0), qn = R(0);
  auto fetch = [&](int n) {
    const long fo = n * a.tstride;
    st_.get(Rows<R>(a.mu + fo, fb));
    if (p1 && ti.own) pn = Rows<R>(p1 + fo, fb).template get<ROWS_NT>(lb, own);
    if (p2 && ti.own) qn = Rows<R>(p2 + fo, fb).template get<ROWS_NT>(lb, own);
  };
  // vr goes where the second tracer will be; with it the first tracer, so that the
  // weights are formed with no rows in flight
  Stager<R, NCH, RING2_NWA> sv(st_);
  sv.get(Rows<R>(vr, fb));
  fetch(ti.n0);
  sv.put(smem_raw + sg.bytes);
  st_.put(smem_raw);
  __syncthreads();
  unsigned row[19];
#pragma unroll
  for (int i = 0; i < 19; ++i) row[i] = (((unsigned)I[R2_PLACEA + i / 4] >> (8 * (i % 4))) & 255u) * sg.pitch;
  RingAdj<R> f;
  ring_adj<sizeof(R) == 4 ? 0 : 18>(m, I, K, a, c, l, f,
                                    [&](int i) { return lds_row<R>(smem_raw + sg.bytes + mb, row[i]); });
  __syncthreads();
  for (int n = ti.n0; n < ti.n1; ++n) {
    const unsigned char *buf = smem_raw + ((n - ti.n0) & 1) * sg.bytes + lb;
    const R mr = lds_row<R>(buf, row[18]);
    const R p = pn, q2 = qn;
    const bool more = n + 1 < ti.n1;
    if (more) fetch(n + 1);
    R mu, nucc;
    const R lq = ring_adj_value(f, mr, mu, nucc, a.dtr, body, k,
                                 [&](int i, unsigned z) { return lds_row<R>(buf, row[i] + z); });
    ring_adj_store(a, h, f, lq, mu, nucc, p, q2, body, k, act && ti.own, n, cb + l);
    if (more) {
      st_.put(smem_raw + ((n + 1 - ti.n0) & 1) * sg.bytes);
      __syncthreads();
    }
  }
}

// ---------------------------------------------------------------- dynamics
// The horizontal advective fluxes of prog_wrt_begs (prog_wrtv_rk.f90:632-661) with their
// face values (fluxes_wrtv, :1022-1081) and gradients (grad_t2d), order 2, no nudging and
// no monotone fluxes, columns of one wave: sums over the faces of mass, thil and the three
// momenta, for k_dyn_w to finish the column with.  k_dyn_grad and the face loop of k_dyn_w,
// which this replaces, wrote eight gradient fields and gathered twelve rows a face.  Per
// field the block stages the rows of its columns' two rings (see Stager), forms the
// gradients of its columns and their first ring, about 2.3 a column, in LDS, and each column
// sums its faces from there.  The expressions and their order are those of k_dyn_grad and
// k_dyn_w, so every sum is the same to the bit.
// Entry e of a block's gradients belongs to wave e mod 16; a wave reads its up to four
// entries at once, 16 lanes each, and broadcasts from there.
// A face's upwind side, distances and places are the same for the four fields: they are
// chosen once, per lane, and a field then costs one value, one gradient and six operations
// a face (choosing per field: 256,002 columns 0.59 ms, now 0.50).  Bound by vector
// instructions (960 a column, 1.6 of 2.0 ms at 1,024,002 columns) and the bytes (5.8 GB, 1.0
// ms there).  ms a launch of the gradient pass and the column kernel
// before, of this and the column kernel now: 256,002 columns of 50 levels in mixed precision
// 0.29 + 1.10, 0.50 + 0.51; 1,024,002 of 60 in FP32 1.16 + 4.21, 2.02 + 1.95; 100,002 of 45
// in FP64 0.27 + 0.77, 0.41 + 0.29.
enum { R2_GWORDS = 16, R2_GENTRIES = WAVE / R2_GWORDS, R2_KD = 30 };
template <class R>
struct Ring2Grad {
  const int *count;      // per block: cells whose gradient is formed
  const int *place;      // per block and entry, 4 words: places of its slots 0..3 and 4..5, its own, 0 (bytes)
  const R *cof;          // per block and entry, 16 words: gxps_coef, gyps_coef of its six slots
  const R *kd;           // nw x R2_KD: dirv, dxps and dyps of this column's side, of the other side
  int gmax;
};
template <class R>
struct alignas(2 * sizeof(R)) GradPair {
  R x, y;
};
template <class R, class RP>
struct DynFlux {
  const R *q[4];         // thil, vxe, vye, vze
  const R *t[4];         // their volume-weighted tendencies, where the sums start
  const R *vmc;
  R *out[4];
  RP *hflx;
};
template <class R, class RP, int NCH>
__global__ __launch_bounds__(RING2_NWF * WAVE, sizeof(R) == 4 ? 8 : 1) void k_dyn_flux(DMesh<R> m, Ring2Tab<R> t,
                                                                                       Ring2Stage sg, Ring2Grad<R> gr,
                                                                                       DynFlux<R, RP> a) {
  NOCONTRACT
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const int blk = xcd_block(blockIdx.x, gridDim.x), wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int w = blk * RING2_NWF + wv, l = lane_id(), k = l + 1, mza = m.mza;
  const bool own = w < m.nw;
  const int c = min(w, m.nw - 1);
  const bool body = k >= 2 && k <= mza;
  const unsigned rowb = (unsigned)(m.ldk * sizeof(R)), fb = field_bytes(m), lb = (unsigned)l * (unsigned)sizeof(R),
                 mine = (unsigned)c * rowb, vb = (unsigned)m.nv * rowb;
  unsigned char *grad = smem_raw + 2 * sg.bytes;
  const RecI I(t.ints, c);
  const RecK<R, R2_KD> K(gr.kd, c);
  Stager<R, NCH, RING2_NWF> st(sg, blk, m.ldk);
  st.get(Rows<R>(a.q[0], fb));
  const int ng = gr.count[blk], mye = wv + (l / R2_GWORDS) * RING2_NWF;
  R gk = R(0);
  int gp = 0;
  if (mye < ng) {
    const long at = (long)blk * gr.gmax + mye;
    gk = gr.cof[at * R2_GWORDS + l % R2_GWORDS];
    gp = gr.place[at * 4 + l % 4];
  }
  // vmca = vmc * arv of the faces (:347-355)
  R vs[6], kx[6], ky[6];
  unsigned qa[6], ga[6];
  {
    const Rows<R> v(a.vmc, vb), ar(m.arv, vb);
    R x[6], y[6];
#pragma unroll
    for (int j = 0; j < 6; ++j) {
      const unsigned f = (unsigned)I[R2_FACE + j] * rowb;
      x[j] = v.get(lb, f);
      y[j] = ar.get(lb, f);
    }
    const int np = I[R2_NPOLY];
#pragma unroll
    for (int j = 0; j < 6; ++j) vs[j] = j < np ? x[j] * y[j] : R(0);
  }
  R tq = Rows<R>(a.t[0], fb).template get<ROWS_NT>(lb, mine);
  st.put(smem_raw);
  // slots in the order and with the signs of k_dyn_w: dirv > 0 adds.  The upwind side, its
  // distances and places are the same for every field.
  RP hflx = RP(0);
  auto place = [&](int i) { return (((unsigned)I[R2_PLACE + i / 4] >> (8 * (i % 4))) & 255u) * sg.pitch; };
  auto gplace = [&](int i) { return (((unsigned)I[R2_GRAD + i / 4] >> (8 * (i % 4))) & 255u) * 2u * sg.pitch; };
#pragma unroll
  for (int j = 0; j < 6; ++j) {
    const R dv = K[j], vm = vs[j];
    const bool sel = (dv < R(0)) ? (vm < R(0)) : !(vm < R(0));
    hflx = dv > R(0) ? hflx + (RP)vm : hflx - (RP)vm;
    vs[j] = dv > R(0) ? vm : -vm;
    kx[j] = sel ? K[18 + j] : K[6 + j];
    ky[j] = sel ? K[24 + j] : K[12 + j];
    qa[j] = (sel ? place(j) : place(18)) + lb;
    ga[j] = (sel ? gplace(j) : gplace(6)) + 2u * lb;
  }
  if (own && body) a.hflx[(long)c * m.ldk + l] = hflx;
  __syncthreads();
#pragma unroll 1
  for (int q = 0; q < 4; ++q) {
    const unsigned char *buf = smem_raw + (q & 1) * sg.bytes;
    R sum = tq;
    if (q < 3) {
      st.get(Rows<R>(a.q[q + 1], fb));
      tq = Rows<R>(a.t[q + 1], fb).template get<ROWS_NT>(lb, mine);
    }
    // gradients (grad_t2d), x and y of a level side by side
#pragma unroll
    for (int i = 0; i < R2_GENTRIES; ++i) {
      const int e = wv + i * RING2_NWF, g0 = i * R2_GWORDS;
      if (e >= ng) break;
      const unsigned p03 = (unsigned)__builtin_amdgcn_readlane(gp, g0), p45 = (unsigned)__builtin_amdgcn_readlane(gp, g0 + 1),
                     po = (unsigned)__builtin_amdgcn_readlane(gp, g0 + 2);
      const R s0 = lds_row<R>(buf + lb, po * sg.pitch);
      R ax = R(0), ay = R(0);
#pragma unroll
      for (int j = 0; j < 6; ++j) {
        const R d = lds_row<R>(buf + lb, (((j < 4 ? p03 : p45) >> (8 * (j & 3))) & 255u) * sg.pitch) - s0;
        ax = ax + lane_word(gk, g0 + j) * d;
        ay = ay + lane_word(gk, g0 + 6 + j) * d;
      }
      if (!body) { ax = R(0); ay = R(0); }
      if (k <= mza) *reinterpret_cast<GradPair<R> *>(grad + (unsigned)e * 2u * sg.pitch + 2u * lb) = {ax, ay};
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 6; ++j) {
      const GradPair<R> g = *reinterpret_cast<const GradPair<R> *>(grad + ga[j]);
      const R f = lds_row<R>(buf, qa[j]) + kx[j] * g.x + ky[j] * g.y;
      sum = sum + vs[j] * f;
    }
    if (own && body) a.out[q][(long)c * m.ldk + l] = sum;
    if (q < 3) {
      st.put(smem_raw + ((q + 1) & 1) * sg.bytes);
      __syncthreads();
    }
  }
}
