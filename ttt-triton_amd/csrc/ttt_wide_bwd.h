// Backward kernels of ttt_wide.h: the readout's gradients and the reverse
// recurrence.
#pragma once

#include "ttt_wide_fwd.h"

namespace ttt {
namespace {

// One (chain, mini-batch): the readout again, then its gradients.  The output
// LayerNorm's backward is a row pass in place of Zb; the hidden slices then
// pass through LDS a second time, each in two halves (before and after dZ1b
// is known), so nine 64 x 64 matrices are enough.
template <typename T, class C> __global__ __launch_bounds__(C::NTH) void wide_bwd_readout_kernel(WideArgs a) {
  constexpr int K = C::K, F = C::F, FF = C::FF, V = C::V, LS = C::LS, LF = C::LF, LK = C::LK, NSL = C::NSL, NT = C::NT;
  using Sl = WideSlot<C>;
  typedef typename VecF<V>::type vf;
  __shared__ __align__(16) float sm[WideReadout<T, C>::LDS];
  const size_t m = blockIdx.x;  // chain * NC + s
  const int h = (int)((m / (size_t)a.NC) % (size_t)a.H);
  float* const slot = a.saved + m * Sl::FLOATS;
  WideReadout<T, C> ro(sm, slot);
  ro.forward(a, m);
  const int w = ro.w, lane = lane_id(), tid = threadIdx.x;
  const WideTile<4> ts = ro.ts;
  const WideTile<C::FT> tf = ro.tf;
  const WideTile<C::KT> tk = ro.tk;
  const f4 zero = f4{0.f, 0.f, 0.f, 0.f};
  const T* const DO = static_cast<const T*>(a.dout) + m * K * F;
  // LayerNorm-parameter partials of the waves' four rows, [2][NW][F]: in W1's
  // place (MLP: staged again below) or X2's (Linear: unused)
  float* const part = C::MLP ? ro.W1 : ro.X2;
  {
    float sd;
    const vf zh = ro.norm(a.eps, sd);
    const vf d = actf<T, V>(ldact<T, V>(DO + (unsigned)(ro.prow * F + ro.pcol)));
    const vf dh = d * ldv<V>(a.ln_w + (size_t)h * F + ro.pcol);
    float m1 = 0.f, m2 = 0.f;
#pragma unroll
    for (int q = 0; q < V; ++q) {
      m1 += dh[q];
      m2 += dh[q] * zh[q];
    }
    m1 = sum_row16(m1) * (1.0f / F);
    m2 = sum_row16(m2) * (1.0f / F);
    stv<V>(ro.Z + ro.prow * LF + ro.pcol, (dh - m1 - zh * m2) * (1.0f / sd));
    vf pw, pb;
#pragma unroll
    for (int q = 0; q < V; ++q) {
      pw[q] = sum_col4(d[q] * zh[q]);
      pb[q] = sum_col4(d[q]);
    }
    if (lane < 16) {
      stv<V>(part + w * F + ro.pcol, pw);
      stv<V>(part + (C::NW + w) * F + ro.pcol, pb);
    }
  }
  __syncthreads();
  if (tid < 2 * F) {  // (2 F <= NTH)
    float t = 0.f;
    const float* p = part + (tid / F) * C::NW * F + tid % F;
#pragma unroll
    for (int q = 0; q < C::NW; ++q) t += p[q * F];
    slot[(tid < F ? Sl::HLW : Sl::HLB) + tid % F] = t;
  }
  f4 deta = zero, da = zero;  // of the wave's K x K tile
  f4 dxq = zero;              // of its K x F tile
  float* const DA = C::MLP ? ro.G2 : ro.W2;  // d(X2b X2^T), then d(XQ XK^T)
  if (C::ALLK || ro.has_k) {
    const f4 dc = wmm_on<WideFree<C>, F, false, true, LF, LF>(zero, ro.Z + 16 * tk.it * LF, ro.G2 + 16 * tk.jt * LF);  // -dC
    deta = -(dc * ((C::MLP ? ro.a2 : ro.a1) + 1.0f));
    da = -(dc * ro.eta);
  }
  if (C::ALLF || ro.has_f) {  // -C^T dZ2b
    const f4 t = wmm_on<WideFree<C>, K, true, false, LK, LF>(zero, ro.C1 + 16 * tf.it, ro.Z + 16 * tf.jt);
    stf4(tf.template at<F>(slot + Sl::HG2), t);
  }
  float cs;
  if constexpr (C::MLP) {
    __syncthreads();
    if (C::ALLK || ro.has_k) {
      stf4(tk.template at<LK>(DA), da);
      stf4(tk.template at<LK>(ro.C1), -(ro.eta * (ro.a1 + 1.0f)));
    }
    f4 dc1 = zero;
#pragma unroll
    for (int sl = 0; sl < NSL; ++sl) {
      f4 x2, g1;
      ro.inner(sl, x2, g1);
      ro.stage_w2(sl);
      stf4(ts.template at<LS>(ro.X2), x2);
      stf4(ts.template at<LS>(ro.XB), ro.xb[sl]);
      __syncthreads();
      f4 dz = wmm_on<WideFree<C>, F, false, true, LF, LF>(zero, ro.Z + 16 * ts.it * LF, ro.W2 + 16 * ts.jt * LF);
      dz = wmm<WideFree<C>, K, false, false, LK, LS>(dz, DA + 16 * ts.it * LK, ro.X2 + 16 * ts.jt);
      dz *= ro.db[sl];
      stf4(ts.template at<FF>(slot + Sl::HX2 + sl * 64), wmm_on<WideFree<C>, K, true, false, LK, LS>(zero, DA + 16 * ts.it, ro.XB + 16 * ts.jt));
#pragma unroll
      for (int n = 0; n < NT; ++n) {
        const int t = w + n * C::NW;
        if (C::ALLT || t < C::TW) {
          const WideTile<C::FT> t2(t);
          f4 dw;
          if (sl == 0 && t2.it == 0) {
            dw = wmm<WideFree<C>, K, true, false, LS, LF, true>(zero, ro.XB, ro.Z + 16 * t2.jt, &cs);
            if (lane < 16) slot[Sl::HST + Sl::B2 + 16 * t2.jt + lane] = cs;
          } else {
            dw = wmm_on<WideFree<C>, K, true, false, LS, LF>(zero, ro.XB + 16 * t2.it, ro.Z + 16 * t2.jt);
          }
          stf4(t2.template at<F>(slot + Sl::HST + Sl::W2 + sl * 64 * F), dw);
        }
      }
      __syncthreads();
      stf4(ts.template at<LS>(ro.XB), dz);
      stf4(ts.template at<LS>(ro.X2), g1);
      ro.stage_w1(sl);
      __syncthreads();
      if (C::ALLF || ro.has_f) dxq = wmm_sl<WideFree<C>, C::S, false, true, LS, LS>(dxq, ro.XB + 16 * tf.it * LS, ro.W1 + 16 * tf.jt * LS);
      if (C::ALLK || ro.has_k) dc1 = wmm_sl<WideFree<C>, C::S, false, true, LS, LS>(dc1, ro.XB + 16 * tk.it * LS, ro.X2 + 16 * tk.jt * LS);
      stf4(ts.template at<FF>(slot + Sl::HG1 + sl * 64), wmm_on<WideFree<C>, K, true, false, LK, LS>(zero, ro.C1 + 16 * ts.it, ro.XB + 16 * ts.jt));
#pragma unroll
      for (int n = 0; n < NT; ++n) {
        const int t = w + n * C::NW;
        if (C::ALLT || t < C::TW) {
          const WideTile<4> t1(t);
          f4 dw;
          if (t1.it == 0) {
            dw = wmm<WideFree<C>, K, true, false, LF, LS, true>(zero, ro.XQ, ro.XB + 16 * t1.jt, &cs);
            if (lane < 16) slot[Sl::HST + Sl::B1 + sl * 64 + 16 * t1.jt + lane] = cs;
          } else {
            dw = wmm_on<WideFree<C>, K, true, false, LF, LS>(zero, ro.XQ + 16 * t1.it, ro.XB + 16 * t1.jt);
          }
          stf4(t1.template at<FF>(slot + Sl::HST + Sl::W1 + sl * 64), dw);
        }
      }
      if (sl + 1 < NSL) __syncthreads();
    }
    if (C::ALLK || ro.has_k) {
      deta -= dc1 * (ro.a1 + 1.0f);
      da = -(dc1 * ro.eta);
      stf4(tk.template at<LK>(DA), da);
    }
  } else {
    dxq = wmm_on<WideFree<C>, F, false, true, LF, LS>(zero, ro.Z + 16 * tf.it * LF, ro.W1 + 16 * tf.jt * LS);
#pragma unroll
    for (int n = 0; n < NT; ++n) {
      const int t = w + n * C::NW;
      if (C::ALLT || t < C::TW) {
        const WideTile<4> t1(t);
        f4 dw;
        if (t1.it == 0) {
          dw = wmm<WideFree<C>, K, true, false, LF, LF, true>(zero, ro.XQ, ro.Z + 16 * t1.jt, &cs);
          if (lane < 16) slot[Sl::HST + Sl::B1 + 16 * t1.jt + lane] = cs;
        } else {
          dw = wmm_on<WideFree<C>, K, true, false, LF, LF>(zero, ro.XQ + 16 * t1.it, ro.Z + 16 * t1.jt);
        }
        stf4(t1.template at<F>(slot + Sl::HST + Sl::W1), dw);
      }
    }
    if (C::ALLK || ro.has_k) stf4(tk.template at<LK>(DA), da);
  }
  // an lr rule sums coef * deta over the rows: through LDS, in the place of a
  // matrix that is dead here (MLP: dZ2b; Linear: XB)
  const bool lr_rule = a.eta_rule == TTT_ETA_LAYER || a.eta_rule == TTT_ETA_CAUSAL;
  float* const DE = C::MLP ? ro.Z : ro.XB;
  if (C::ALLK || ro.has_k) {
    const int i = tk.row(), j = tk.col();
    if (lr_rule) {
      f4 t;
#pragma unroll
      for (int q = 0; q < 4; ++q) t[q] = deta[q] * wide_eta_coef<K>(a.eta_rule, i, j + q);
      stf4(DE + i * LK + j, t);
    } else if (i == K - 1) {
      stf4(slot + Sl::HDE + j, deta);  // (wide_bwd_state adds the update's term and stores the row)
    } else if (a.eta_rule == TTT_ETA_DENSE) {
      st4(static_cast<T*>(a.deta) + (m * K + i) * K + j, deta);
    } else {
      stf4(static_cast<float*>(a.deta) + (m * K + i) * K + j, deta);
    }
  }
  __syncthreads();
  if (C::ALLF || ro.has_f) {
    dxq = wmm<WideFree<C>, K, false, false, LK, LF>(dxq, DA + 16 * tf.it * LK, ro.XK + 16 * tf.jt);
    st4(tf.template at<F>(static_cast<T*>(a.dXQ) + m * K * F), dxq + frag_to_f4(ldraw4(tf.template at<F>(DO))));
    stf4(tf.template at<F>(slot + Sl::HXK), wmm_on<WideFree<C>, K, true, false, LK, LF>(zero, DA + 16 * tf.it, ro.XQ + 16 * tf.jt));
  }
  if (lr_rule && tid < K) {
    float t = 0.f;
#pragma unroll 8
    for (int i = 0; i < K; ++i) t += DE[i * LK + tid];
    slot[Sl::HDE + tid] = t;
  }
}

// Per chain, the mini-batches in reverse: the gradient through the update,
// carrying dL/d(state) in registers (and, slice by slice, in LDS).
template <typename T, class C> __global__ __launch_bounds__(C::NTH) void wide_bwd_state_kernel(WideArgs a) {
  constexpr int K = C::K, F = C::F, FF = C::FF, V = C::V, LS = C::LS, LF = C::LF, NSL = C::NSL, NT = C::NT;
  constexpr bool MLP = C::MLP;
  using Sl = WideSlot<C>;
  typedef typename VecF<V>::type vf;
  typedef typename VecT<T, V>::type vt;
  __shared__ __align__(16) float sm[9 * C::SLOT];
  __shared__ __align__(16) float db1s[FF], db2s[F];
  __shared__ float dep[8][K];
  float* const XKs = sm;
  float* const G2s = sm + C::SLOT;
  float* const DGs = sm + 2 * C::SLOT;   // dG2, then dZ2 in place
  float* const DTs = sm + 3 * C::SLOT;   // d target
  float* const DW1s = sm + 4 * C::SLOT;  // dW1 of a slice, then dP, then dZ1
  float* const DW2s = sm + 5 * C::SLOT;
  float* const X2s = sm + 6 * C::SLOT;
  float* const G1s = sm + 7 * C::SLOT;   // G1 of a slice, then W1
  float* const W2s = sm + 8 * C::SLOT;
  const size_t chain = blockIdx.x;
  const int h = (int)(chain % (size_t)a.H), NC = a.NC;
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = wide_wave<C>();
  const int prow = tid >> 4, pcol = (tid & 15) * V;
  const unsigned po = (unsigned)(prow * F + pcol);
  const vf lw = ldv<V>(a.ln_w + (size_t)h * F + pcol), lb = ldv<V>(a.ln_b + (size_t)h * F + pcol);
  const WideTile<4> ts(w);
  const WideTile<C::FT> tf(w);
  const bool has_f = C::f_tile(w);
  float* const slot0 = a.saved + chain * NC * (size_t)Sl::FLOATS;
  const f4 zero = f4{0.f, 0.f, 0.f, 0.f};
  f4 dw1[NSL][NT], dw2[MLP ? NSL : 1][NT];
#pragma unroll
  for (int sl = 0; sl < NSL; ++sl)
#pragma unroll
    for (int n = 0; n < NT; ++n) {
      dw1[sl][n] = zero;
      if constexpr (MLP) dw2[sl][n] = zero;
    }
  vf accw, accb;  // LayerNorm-parameter gradients of this thread's row part
#pragma unroll
  for (int q = 0; q < V; ++q) accw[q] = accb[q] = 0.f;
  float hln = 0.f;  // thread < 2 F: the readout's LayerNorm-parameter terms
  for (int i = tid; i < FF; i += C::NTH) db1s[i] = 0.f;
  for (int i = tid; i < F; i += C::NTH) db2s[i] = 0.f;
  for (int i = tid; i < 8 * K; i += C::NTH) (&dep[0][0])[i] = 0.f;
  const size_t row00 = chain * NC * K;
  const T *const XK = static_cast<const T*>(a.XK), *const XV = static_cast<const T*>(a.XV);
  // the first products' operands, requested a mini-batch ahead
  size_t m = chain * NC + NC - 1;
  float* slot = slot0 + (size_t)(NC - 1) * Sl::FLOATS;
  vt rxk = ldact<T, V>(XK + m * K * F + po);
  vf rg2 = ldv<V>(slot + Sl::G2 + po);
  f4 rz = zero, rp = zero;
  if constexpr (MLP) {
    rz = ldf4(ts.template at<FF>(slot + Sl::Z1));
    rp = ldf4(ts.template at<FF>(slot + Sl::P));
  }

  const int lane0 = lane;
  for (int s = NC - 1; s >= 0; --s) {
    m = chain * NC + s;
    if constexpr (C::PIN) m = pinned_index(m);
    slot = a.saved + m * Sl::FLOATS;
    const int lane = C::PIN ? pinned(lane0) : lane0, tid = 64 * w + lane;
    const int prow = tid >> 4, pcol = (tid & 15) * V;
    const unsigned po = (unsigned)(prow * F + pcol);
    const WideTile<4> ts(w, lane);
    const WideTile<C::FT> tf(w, lane);
    const vt rxv = ldact<T, V>(XV + m * K * F + po);
    const vf zh = ldv<V>(slot + Sl::ZH + po);
    const float sd = (slot + Sl::SIG)[(unsigned)prow];
    const unsigned es = wide_eta_last_raw<T, K>(a, m, ts.row());
    const unsigned ef = C::FT == 4 ? es : has_f ? wide_eta_last_raw<T, K>(a, m, C::f_token(w, lane)) : 0u;
    if (tid < 2 * F) hln += (slot + Sl::HLW)[(unsigned)tid];  // (HLB follows HLW)
    const vf xk = actf<T, V>(rxk), g2 = rg2;
    stv<V>(XKs + prow * LF + pcol, xk);
    stv<V>(G2s + prow * LF + pcol, g2);
    const float e_s = wide_eta_last_val<T, K>(a, es), e_f = wide_eta_last_val<T, K>(a, ef);
    f4 dxk = zero, dg2 = zero, t2 = zero;  // K x F tile
    f4 dz1a[MLP ? NSL : 1], dx2[MLP ? NSL : 1], d1[MLP ? NSL : 1];
    auto stage_w1 = [&](int sl) {  // W1 of the state entering the mini-batch, in G1's place
#pragma unroll
      for (int n = 0; n < NT; ++n) {
        const int t = w + n * C::NW;
        if (C::ALLT || t < C::TW) {
          const WideTile<4> t1(t, lane);
          stf4(t1.template at<LS>(G1s), ldf4(t1.template at<FF>(slot + Sl::W1 + sl * 64)));
        }
      }
    };
    auto stage_w2 = [&](int sl) {
#pragma unroll
      for (int n = 0; n < NT; ++n) {
        const int t = w + n * C::NW;
        if (C::ALLT || t < C::TW) {
          const WideTile<C::FT> t2t(t, lane);
          stf4(t2t.template at<LF>(W2s), ldf4(t2t.template at<F>(slot + Sl::W2 + sl * 64 * F)));
        }
      }
    };
    if constexpr (MLP) {
#pragma unroll
      for (int sl = 0; sl < NSL; ++sl) {
        auto ld = [&](int off) { return ldf4(ts.template at<FF>(slot + off + sl * 64)); };
        const f4 hg1 = ld(Sl::HG1), hx2 = ld(Sl::HX2);
        const f4 z = sl == 0 ? rz : ld(Sl::Z1), p = sl == 0 ? rp : ld(Sl::P);
        f4 x2, dd1;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          float y, dy, ddy;
          gelu_all(z[q], y, dy, ddy);
          x2[q] = y;
          d1[sl][q] = dy;
          dd1[q] = ddy;
        }
        const f4 g1 = p * d1[sl];
#pragma unroll
        for (int n = 0; n < NT; ++n) {
          const int t = w + n * C::NW;
          if (C::ALLT || t < C::TW) {
            const WideTile<4> t1(t, lane);
            const WideTile<C::FT> t2t(t, lane);
            stf4(t1.template at<LS>(DW1s), dw1[sl][n]);
            stf4(t2t.template at<LF>(DW2s), dw2[sl][n]);
          }
        }
        stf4(ts.template at<LS>(X2s), x2);
        stf4(ts.template at<LS>(G1s), g1);
        stage_w2(sl);
        __syncthreads();
        // through the update W1' = W1 - XK^T (e G1), b1' = b1 - G1^T e
        const f4 t = wmm_on<C, F, false, false, LF, LS>(ldf4(db1s + sl * 64 + ts.col()), XKs + 16 * ts.it * LF,
                                                  DW1s + 16 * ts.jt);
        const f4 tg = t * g1;
        const float dpart = sum_col4((tg[0] + tg[1]) + (tg[2] + tg[3]));
        if (lane < 16) dep[ts.jt][ts.row()] = (sl == 0 ? 0.f : dep[ts.jt][ts.row()]) - dpart;
        const f4 dg1 = hg1 - t * e_s;
        dz1a[sl] = dg1 * p * dd1;
        dx2[sl] = hx2 - wmm_on<C, F, false, true, LF, LF>(zero, G2s + 16 * ts.it * LF, DW2s + 16 * ts.jt * LF) * e_s;
        if (has_f) {
          t2 = wmm_sl<C, C::S, false, false, LS, LF>(t2, X2s + 16 * tf.it * LS, DW2s + 16 * tf.jt);
          dxk = wmm_sl<C, C::S, false, true, LS, LS>(dxk, G1s + 16 * tf.it * LS, DW1s + 16 * tf.jt * LS);
        }
        __syncthreads();
        stf4(ts.template at<LS>(DW1s), dg1 * d1[sl]);  // dP
        if constexpr (NSL == 1) stage_w1(0);
        __syncthreads();
        if (has_f) dg2 = wmm_sl<C, C::S, false, false, LS, LF>(dg2, DW1s + 16 * tf.it * LS, W2s + 16 * tf.jt);
#pragma unroll
        for (int n = 0; n < NT; ++n) {
          const int tt = w + n * C::NW;
          if (C::ALLT || tt < C::TW) {
            const WideTile<C::FT> t2t(tt, lane);
            dw2[sl][n] = wmm<C, K, true, false, LS, LF>(dw2[sl][n], DW1s + 16 * t2t.it, G2s + 16 * t2t.jt);
          }
        }
        if (sl + 1 < NSL) __syncthreads();
      }
    } else {
#pragma unroll
      for (int n = 0; n < NT; ++n) {
        const int t = w + n * C::NW;
        if (C::ALLT || t < C::TW) {
          const WideTile<4> t1(t, lane);
          stf4(t1.template at<LS>(DW1s), dw1[0][n]);
        }
      }
      stage_w1(0);
      __syncthreads();
      t2 = wmm_on<C, F, false, false, LF, LS>(t2, XKs + 16 * tf.it * LF, DW1s + 16 * tf.jt);
      dxk = wmm_on<C, F, false, true, LF, LS>(dxk, G2s + 16 * tf.it * LF, DW1s + 16 * tf.jt * LS);
    }
    if (has_f) {
      t2 += ldf4((MLP ? db2s : db1s) + tf.col());
      const f4 tg = t2 * ldf4(tf.template at<LF>(G2s));
      const float dpart = sum_col4((tg[0] + tg[1]) + (tg[2] + tg[3]));
      if (lane < 16) dep[4 + tf.jt][tf.row()] = -dpart;
      stf4(tf.template at<LF>(DGs), dg2 + ldf4(tf.template at<F>(slot + Sl::HG2)) - t2 * e_f);
      dxk = ldf4(tf.template at<F>(slot + Sl::HXK)) - dxk * e_f;
    }
    // the next (earlier) mini-batch's first operands
    if (s > 0) {
      const float* q = slot - Sl::FLOATS;
      rxk = ldact<T, V>(XK + (m - 1) * K * F + po);
      rg2 = ldv<V>(q + Sl::G2 + po);
      if constexpr (MLP) {
        rz = ldf4(ts.template at<FF>(q + Sl::Z1));
        rp = ldf4(ts.template at<FF>(q + Sl::P));
      }
    }
    __syncthreads();
    {  // backward of the LayerNorm fused with the L2 loss's gradient
      const float rs = 1.0f / sd, inv = rs * (1.0f / F);
      vf qv = ldv<V>(DGs + prow * LF + pcol);
      const vf rr = lw * zh + lb - (actf<T, V>(rxv) - xk);
      const vf gx = lw * rr;
      float S2 = 0.f, Q1 = 0.f, Q2 = 0.f, QG = 0.f;
#pragma unroll
      for (int q = 0; q < V; ++q) {
        S2 += gx[q] * zh[q];
        Q1 += qv[q];
        Q2 += qv[q] * zh[q];
        QG += qv[q] * g2[q];
      }
      S2 = sum_row16(S2);
      Q1 = sum_row16(Q1);
      Q2 = sum_row16(Q2);
      QG = sum_row16(QG);
      const vf dg = ((float)F * qv - Q1 - zh * Q2) * inv;
      const vf dt = -(dg * lw);
      accw += dg * (rr + lw * zh);
      accb += dg * lw;
      const vf dxh = (-qv * S2 - gx * Q2) * inv + dg * lw * lw;
      float m1 = 0.f, m2 = 0.f;
#pragma unroll
      for (int q = 0; q < V; ++q) {
        m1 += dxh[q];
        m2 += dxh[q] * zh[q];
      }
      m1 = sum_row16(m1) * (1.0f / F);
      m2 = sum_row16(m2) * (1.0f / F);
      stv<V>(DGs + prow * LF + pcol, (dxh - m1 - zh * m2) * rs - zh * (QG * rs * (1.0f / F)));
      stv<V>(DTs + prow * LF + pcol, dt);
      stact<T, V>(static_cast<T*>(a.dXV) + m * K * F + po, dt);
    }
    if (tid < K) {  // deta's last row (dlr): the readout's terms and the update's
      float d = 0.f;
#pragma unroll
      for (int q = 0; q < 8; ++q) d += dep[q][tid];
      const float hd = (slot + Sl::HDE)[(unsigned)tid];
      if (a.eta_rule == TTT_ETA_DENSE)
        stact<T, 1>(static_cast<T*>(a.deta) + (m * K + (K - 1)) * K + tid, typename VecF<1>::type(hd + d));
      else if (a.eta_rule == TTT_ETA_DENSE_F32)
        static_cast<float*>(a.deta)[(m * K + (K - 1)) * K + tid] = hd + d;
      else
        static_cast<float*>(a.deta)[m * K + tid] = hd + d * (1.0f / (float)K);
    }
    __syncthreads();
    float cs;
    if constexpr (MLP) {
#pragma unroll
      for (int sl = 0; sl < NSL; ++sl) {
        if constexpr (NSL > 1) {
          const f4 z = ldf4(ts.template at<FF>(slot + Sl::Z1 + sl * 64));
          f4 x2;
#pragma unroll
          for (int q = 0; q < 4; ++q) x2[q] = gelu_tanh(z[q]);
          stf4(ts.template at<LS>(X2s), x2);
          stage_w1(sl);
          stage_w2(sl);
          __syncthreads();
        }
        const f4 dx = wmm<C, F, false, true, LF, LF>(dx2[sl], DGs + 16 * ts.it * LF, W2s + 16 * ts.jt * LF);
        stf4(ts.template at<LS>(DW1s), dz1a[sl] + dx * d1[sl]);  // dZ1
#pragma unroll
        for (int n = 0; n < NT; ++n) {
          const int t = w + n * C::NW;
          if (C::ALLT || t < C::TW) {
            const WideTile<C::FT> t2t(t, lane);
            const f4 hw = ldf4(t2t.template at<F>(slot + Sl::HST + Sl::W2 + sl * 64 * F));
            if (sl == 0 && t2t.it == 0) {
              dw2[sl][n] = wmm<C, K, true, false, LS, LF, true>(dw2[sl][n], X2s, DGs + 16 * t2t.jt, &cs);
              if (lane < 16) db2s[16 * t2t.jt + lane] += cs + (slot + Sl::HST + Sl::B2 + 16 * t2t.jt)[(unsigned)lane];
            } else {
              dw2[sl][n] = wmm<C, K, true, false, LS, LF>(dw2[sl][n], X2s + 16 * t2t.it, DGs + 16 * t2t.jt);
            }
            dw2[sl][n] += hw;
          }
        }
        __syncthreads();
        if (has_f) dxk = wmm<C, C::S, false, true, LS, LS>(dxk, DW1s + 16 * tf.it * LS, G1s + 16 * tf.jt * LS);
#pragma unroll
        for (int n = 0; n < NT; ++n) {
          const int t = w + n * C::NW;
          if (C::ALLT || t < C::TW) {
            const WideTile<4> t1(t, lane);
            const f4 hw = ldf4(t1.template at<FF>(slot + Sl::HST + Sl::W1 + sl * 64));
            if (t1.it == 0) {
              dw1[sl][n] = wmm<C, K, true, false, LF, LS, true>(dw1[sl][n], XKs, DW1s + 16 * t1.jt, &cs);
              const int c = sl * 64 + 16 * t1.jt + lane;
              if (lane < 16) db1s[c] += cs + slot[Sl::HST + Sl::B1 + c];
            } else {
              dw1[sl][n] = wmm<C, K, true, false, LF, LS>(dw1[sl][n], XKs + 16 * t1.it, DW1s + 16 * t1.jt);
            }
            dw1[sl][n] += hw;
          }
        }
        if (sl + 1 < NSL) __syncthreads();
      }
    } else {
      dxk = wmm<C, F, false, true, LF, LS>(dxk, DGs + 16 * tf.it * LF, G1s + 16 * tf.jt * LS);
#pragma unroll
      for (int n = 0; n < NT; ++n) {
        const int t = w + n * C::NW;
        if (C::ALLT || t < C::TW) {
          const WideTile<4> t1(t, lane);
          const f4 hw = ldf4(t1.template at<F>(slot + Sl::HST + Sl::W1));
          if (t1.it == 0) {
            dw1[0][n] = wmm<C, K, true, false, LF, LF, true>(dw1[0][n], XKs, DGs + 16 * t1.jt, &cs);
            const int c = 16 * t1.jt + lane;
            if (lane < 16) db1s[c] += cs + slot[Sl::HST + Sl::B1 + c];
          } else {
            dw1[0][n] = wmm<C, K, true, false, LF, LF>(dw1[0][n], XKs + 16 * t1.it, DGs + 16 * t1.jt);
          }
          dw1[0][n] += hw;
        }
      }
    }
    if (has_f) {
      const f4 dt = ldf4(tf.template at<LF>(DTs));
      st4(tf.template at<F>(static_cast<T*>(a.dXK) + m * K * F), dxk - dt);
    }
    __syncthreads();
  }
#pragma unroll
  for (int sl = 0; sl < NSL; ++sl)
#pragma unroll
    for (int n = 0; n < NT; ++n) {
      const int t = w + n * C::NW;
      if (C::ALLT || t < C::TW) {
        const WideTile<4> t1(t);
        stf4(t1.template at<FF>(a.dW1 + chain * F * FF + sl * 64), dw1[sl][n]);
        if constexpr (MLP) {
          const WideTile<C::FT> t2t(t);
          stf4(t2t.template at<F>(a.dW2 + (chain * FF + sl * 64) * F), dw2[sl][n]);
        }
      }
    }
  for (int i = tid; i < FF; i += C::NTH) a.db1[chain * FF + i] = db1s[i];
  if constexpr (MLP)
    for (int i = tid; i < F; i += C::NTH) a.db2[chain * F + i] = db2s[i];
  // LayerNorm-parameter gradients: the rows of each wave, then the waves
  vf pw, pb;
#pragma unroll
  for (int q = 0; q < V; ++q) {
    pw[q] = sum_col4(accw[q]);
    pb[q] = sum_col4(accb[q]);
  }
  if (lane < 16) {
    stv<V>(sm + w * F + pcol, pw);
    stv<V>(sm + (C::NW + w) * F + pcol, pb);
  }
  __syncthreads();
  if (tid < 2 * F) {
    float t = hln;
    const float* p = sm + (tid / F) * C::NW * F + tid % F;
#pragma unroll
    for (int q = 0; q < C::NW; ++q) t += p[q * F];
    (tid < F ? a.dln_w : a.dln_b)[chain * F + tid % F] = t;
  }
}

}  // namespace
}  // namespace ttt
