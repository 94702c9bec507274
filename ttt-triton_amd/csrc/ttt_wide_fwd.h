// Forward kernels of ttt_wide.h: the state recurrence and the readout.
#pragma once

#include "ttt_wide.h"

namespace ttt {
namespace {

// The normalised row of a thread group's 16 lanes (V features each), from
// z = x + bias: returns (z - mean) / sd and sd.
template <int V, int F>
__device__ __forceinline__ typename VecF<V>::type wide_ln_row(typename VecF<V>::type z, float eps, float& sd) {
  float acc = 0.f;
#pragma unroll
  for (int q = 0; q < V; ++q) acc += z[q];
  z -= sum_row16(acc) * (1.0f / F);
  acc = 0.f;
#pragma unroll
  for (int q = 0; q < V; ++q) acc += z[q] * z[q];
  sd = sqrtf(sum_row16(acc) * (1.0f / F) + eps);
  return z * (1.0f / sd);
}

// Where the state after mini-batch s goes (null: nowhere): the next slot's
// state, a checkpoint, a memo snapshot, the final state.
struct WideStateDst {
  float *W1, *b1, *W2, *b2;
};

// Per chain: the recurrence.  LDS: XK twice (the next mini-batch's is staged
// while the last update still reads this one's), G2, -e G2, -e G1, X2, W1, W2
// (of one hidden slice; with several slices the state lives in registers and
// its slices pass through LDS, W2 and X2 in two alternating places, so that
// one barrier separates a slice's writes from its reads).
template <typename T, class C> __global__ __launch_bounds__(C::NTH) void wide_fwd_state_kernel(WideArgs a) {
  constexpr int K = C::K, F = C::F, FF = C::FF, V = C::V, LS = C::LS, LF = C::LF, NSL = C::NSL, NT = C::NT;
  constexpr bool MLP = C::MLP;
  using Sl = WideSlot<C>;
  __shared__ __align__(16) float sm[9 * C::SLOT];
  __shared__ __align__(16) float b1s[FF], b2s[F];
  float* const G2s = sm + 2 * C::SLOT;  // (sm, sm + SLOT: XK of even and odd mini-batches)
  float* const U2s = sm + 3 * C::SLOT;
  float* const W1s = sm + 4 * C::SLOT;
  float* const X2s = sm + 5 * C::SLOT;
  float* const U1s = sm + 6 * C::SLOT;
  float* const W2s = sm + 7 * C::SLOT;  // and sm + 8 SLOT: odd slices
  const size_t chain = blockIdx.x;
  const int h = (int)(chain % (size_t)a.H), NC = a.NC;
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = wide_wave<C>();
  // row pass: this thread's token row and features
  const int prow = tid >> 4, pcol = (tid & 15) * V;
  const unsigned po = (unsigned)(prow * F + pcol);
  typedef typename VecF<V>::type vf;
  const vf lw = ldv<V>(a.ln_w + (size_t)h * F + pcol), lb = ldv<V>(a.ln_b + (size_t)h * F + pcol);
  const WideTile<4> ts(w);        // its K x 64 tile
  const WideTile<C::FT> tf(w);    // its K x F tile
  const bool has_f = C::f_tile(w);
  const int NK = (NC + a.G - 1) / a.G, NS = (NC + a.M - 1) / a.M;
  float* const slot0 = a.saved + chain * NC * a.slot_stride;

  const size_t ic = chain % (size_t)a.NI;
  f4 w1[NSL][NT], w2[NSL][NT];
#pragma unroll
  for (int sl = 0; sl < NSL; ++sl)
#pragma unroll
    for (int n = 0; n < NT; ++n) {
      const int t = w + n * C::NW;
      if (C::ALLT || t < C::TW) {
        const WideTile<4> t1(t);
        w1[sl][n] = ldf4(t1.template at<FF>(a.W1_init + ic * F * FF + sl * 64));
        if constexpr (MLP) {
          const WideTile<C::FT> t2(t);
          w2[sl][n] = ldf4(t2.template at<F>(a.W2_init + (ic * FF + sl * 64) * F));
        }
      }
    }
  for (int i = tid; i < FF; i += C::NTH) b1s[i] = a.b1_init[ic * FF + i];
  if (MLP)
    for (int i = tid; i < F; i += C::NTH) b2s[i] = a.b2_init[ic * F + i];

  // destination i of the state entering mini-batch s (s = NC: the final one):
  // the next slot, a checkpoint, the final state, a memo snapshot.  The
  // checkpoints' and snapshots' next indexes and the mini-batches left until
  // them are counted (a division per use was a tenth of the step).
  int ck = 0, ck_in = 0, mk = 0, mk_in = 1;
  auto dst = [&](int i, int s) {
    auto at = [](float* p, size_t k, size_t n) { return p != nullptr ? p + k * n : nullptr; };
    WideStateDst d{nullptr, nullptr, nullptr, nullptr};
    if (i == 0) {
      // (a store on every path, so that the waits for loads can count past it:
      // after the last mini-batch too)
      float* q = s < NC ? slot0 + s * a.slot_stride : a.fin + chain * a.fin_stride;
      d = WideStateDst{q + Sl::W1, q + Sl::B1, q + Sl::W2, q + Sl::B2};
    } else if (i == 1 && s < NC && ck_in == 0) {
      const size_t k = chain * NK + ck;
      d = WideStateDst{at(a.W1_ckpt, k, F * FF), at(a.b1_ckpt, k, FF), at(a.W2_ckpt, k, FF * F), at(a.b2_ckpt, k, F)};
    } else if (i == 2 && s == NC) {
      d = WideStateDst{at(a.W1_last, chain, F * FF), at(a.b1_last, chain, FF), at(a.W2_last, chain, FF * F),
                       at(a.b2_last, chain, F)};
    } else if (i == 3 && a.W1_memo != nullptr && mk_in == 0) {
      const size_t k = chain * NS + mk;
      d = WideStateDst{at(a.W1_memo, k, F * FF), at(a.b1_memo, k, FF), at(a.W2_memo, k, FF * F), at(a.b2_memo, k, F)};
    }
    return d;
  };
  auto next_dst = [&]() {  // s -> s + 1
    if (--ck_in < 0) {
      ck_in = a.G - 1;
      ++ck;
    }
    if (--mk_in < 0) {
      mk_in = a.M - 1;
      ++mk;
    }
  };
  auto put_w = [&](int s, int sl) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const WideStateDst d = dst(i, s);
#pragma unroll
      for (int n = 0; n < NT; ++n) {
        const int t = w + n * C::NW;
        if (C::ALLT || t < C::TW) {
          const WideTile<4> t1(t);
          const WideTile<C::FT> t2(t);
          if (i == 0 || d.W1 != nullptr) stf4(t1.template at<FF>(d.W1 + sl * 64), w1[sl][n]);
          if constexpr (MLP)
            if (i == 0 || d.W2 != nullptr) stf4(t2.template at<F>(d.W2 + sl * 64 * F), w2[sl][n]);
        }
      }
    }
  };
  auto stage_w1 = [&](int sl) {
#pragma unroll
    for (int n = 0; n < NT; ++n) {
      const int t = w + n * C::NW;
      if (C::ALLT || t < C::TW) {
        const WideTile<4> t1(t);
        stf4(t1.template at<LS>(W1s), w1[sl][n]);
      }
    }
  };
  auto stage_w2 = [&](int sl) {
#pragma unroll
    for (int n = 0; n < NT; ++n) {
      const int t = w + n * C::NW;
      if (C::ALLT || t < C::TW) {
        const WideTile<C::FT> t2(t);
        stf4(t2.template at<LF>(W2s + (sl & 1) * C::SLOT), w2[sl][n]);
      }
    }
  };

#pragma unroll
  for (int sl = 0; sl < NSL; ++sl) put_w(0, sl);
  __syncthreads();  // b1s, b2s
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const WideStateDst d = dst(i, 0);
    if (d.b1 != nullptr)
      for (int j = tid; j < FF; j += C::NTH) d.b1[j] = b1s[j];
    if (MLP && d.b2 != nullptr)
      for (int j = tid; j < F; j += C::NTH) d.b2[j] = b2s[j];
  }
  if constexpr (NSL == 1) {
    stage_w1(0);
    if constexpr (MLP) stage_w2(0);
  }

  const T* const XK = static_cast<const T*>(a.XK);
  const T* const XV = static_cast<const T*>(a.XV);
  typedef typename VecT<T, V>::type vt;
  const size_t row00 = chain * NC * K;  // the chain's first token row
  vt rxk = ldact<T, V>(XK + row00 * F + po), rxv = ldact<T, V>(XV + row00 * F + po);
  unsigned ep = wide_eta_last_raw<T, K>(a, chain * NC, prow), es = wide_eta_last_raw<T, K>(a, chain * NC, ts.row());

  vf xk = actf<T, V>(rxk), tgt = actf<T, V>(rxv) - xk;
  float e_p = wide_eta_last_val<T, K>(a, ep), e_s = wide_eta_last_val<T, K>(a, es);
  stv<V>(sm + prow * LF + pcol, xk);

  for (int s = 0; s < NC; ++s) {
    float* const XKs = sm + (s & 1) * C::SLOT;
    float* const slot = slot0 + s * a.slot_stride;
    next_dst();
    f4 x2[MLP ? NSL : 1], d1[MLP ? NSL : 1];
    f4 z2 = f4{0.f, 0.f, 0.f, 0.f};
    if constexpr (MLP) {
#pragma unroll
      for (int sl = 0; sl < NSL; ++sl) {
        if constexpr (NSL > 1) {
          stage_w1(sl);
          stage_w2(sl);
        }
        __syncthreads();
        f4 z = wmm_on<C, F, false, false, LF, LS>(ldf4(b1s + sl * 64 + ts.col()), XKs + 16 * ts.it * LF, W1s + 16 * ts.jt);
        stf4(ts.template at<FF>(slot + Sl::Z1 + sl * 64), z);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          float y, dy;
          gelu_fwd_bwd(z[q], y, dy);
          x2[sl][q] = y;
          d1[sl][q] = dy;
        }
        stf4(ts.template at<LS>(X2s), x2[sl]);
        __syncthreads();
        if (has_f)
          z2 = wmm_sl<C, C::S, false, false, LS, LF>(z2, X2s + 16 * tf.it * LS, W2s + (sl & 1) * C::SLOT + 16 * tf.jt);
      }
    } else {
      __syncthreads();
      z2 = wmm_on<C, F, false, false, LF, LS>(z2, XKs + 16 * tf.it * LF, W1s + 16 * tf.jt);
    }
    if (has_f) stf4(tf.template at<LF>(G2s), z2);
    // the next mini-batch's inputs are requested here and used after its barrier
    if (s + 1 < NC) {
      const size_t row = row00 + (size_t)(s + 1) * K;
      rxk = ldact<T, V>(XK + row * F + po);
      rxv = ldact<T, V>(XV + row * F + po);
      ep = wide_eta_last_raw<T, K>(a, chain * NC + s + 1, prow);
      es = wide_eta_last_raw<T, K>(a, chain * NC + s + 1, ts.row());
    }
    __syncthreads();
    {  // LayerNorm fused with the L2 loss's gradient, one row per 16 threads
      float sd;
      const vf z = ldv<V>(G2s + prow * LF + pcol) + ldv<V>((MLP ? b2s : b1s) + pcol);
      const vf xh = wide_ln_row<V, F>(z, a.eps, sd);
      vf gr = lw * (lw * xh + lb - tgt);
      float s1 = 0.f, s2 = 0.f;
#pragma unroll
      for (int q = 0; q < V; ++q) {
        s1 += gr[q];
        s2 += gr[q] * xh[q];
      }
      s1 = sum_row16(s1) * (1.0f / F);
      s2 = sum_row16(s2) * (1.0f / F);
      gr = (gr - s1 - xh * s2) * (1.0f / sd);
      stv<V>(G2s + prow * LF + pcol, gr);
      stv<V>(U2s + prow * LF + pcol, gr * -e_p);
      stv<V>(slot + Sl::G2 + po, gr);
      stv<V>(slot + Sl::ZH + po, xh);
      if ((tid & 15) == 0) (slot + Sl::SIG)[(unsigned)prow] = sd;
    }
    // the next mini-batch's inputs arrive before this one's state is stored:
    // a wait for them placed after those stores would wait for the stores too
    vf tgt_n = tgt;
    float e_pn = 0.f, e_sn = 0.f;
    auto take_next = [&]() {
      if (s + 1 < NC) {
        xk = actf<T, V>(rxk);
        tgt_n = actf<T, V>(rxv) - xk;
        e_pn = wide_eta_last_val<T, K>(a, ep);
        e_sn = wide_eta_last_val<T, K>(a, es);
        stv<V>(sm + ((s + 1) & 1) * C::SLOT + prow * LF + pcol, xk);
      }
    };
    float cs;
    auto bias = [&](float* bs, int c, bool second) {  // column sums of -e G onto a bias
      if (lane < 16) {
        const float v = bs[c + lane] + cs;
        bs[c + lane] = v;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const WideStateDst d = dst(i, s + 1);
          float* const p = second ? d.b2 : d.b1;
          if (i == 0 || p != nullptr) p[c + lane] = v;
        }
      }
    };
    if constexpr (MLP) {
#pragma unroll
      for (int sl = 0; sl < NSL; ++sl) {
        float* const x2s = (sl & 1) ? W1s : X2s;
        float* const w2s = W2s + (sl & 1) * C::SLOT;
        if constexpr (NSL > 1) {
          stage_w2(sl);
          stf4(ts.template at<LS>(x2s), x2[sl]);
        }
        __syncthreads();
        const f4 p = wmm_on<C, F, false, true, LF, LF>(f4{0.f, 0.f, 0.f, 0.f}, G2s + 16 * ts.it * LF, w2s + 16 * ts.jt * LF);
        stf4(ts.template at<FF>(slot + Sl::P + sl * 64), p);
        stf4(ts.template at<LS>(U1s), p * d1[sl] * -e_s);
        __syncthreads();
#pragma unroll
        for (int n = 0; n < NT; ++n) {
          const int t = w + n * C::NW;
          if (C::ALLT || t < C::TW) {
            const WideTile<4> t1(t);
            const WideTile<C::FT> t2(t);
            if (t1.it == 0) {
              w1[sl][n] = wmm<C, K, true, false, LF, LS, true>(w1[sl][n], XKs, U1s + 16 * t1.jt, &cs);
              bias(b1s, sl * 64 + 16 * t1.jt, false);
            } else {
              w1[sl][n] = wmm<C, K, true, false, LF, LS>(w1[sl][n], XKs + 16 * t1.it, U1s + 16 * t1.jt);
            }
            if (sl == 0 && t2.it == 0) {
              w2[sl][n] = wmm<C, K, true, false, LS, LF, true>(w2[sl][n], x2s, U2s + 16 * t2.jt, &cs);
              bias(b2s, 16 * t2.jt, true);
            } else {
              w2[sl][n] = wmm<C, K, true, false, LS, LF>(w2[sl][n], x2s + 16 * t2.it, U2s + 16 * t2.jt);
            }
          }
        }
        if (sl == 0) take_next();
        put_w(s + 1, sl);
        if constexpr (NSL == 1) {
          stage_w1(0);
          stage_w2(0);
        }
      }
      if constexpr (NSL > 1) __syncthreads();  // the last slice's X2 is read where W1's first slice goes
    } else {
      __syncthreads();
#pragma unroll
      for (int n = 0; n < NT; ++n) {
        const int t = w + n * C::NW;
        if (C::ALLT || t < C::TW) {
          const WideTile<4> t1(t);
          if (t1.it == 0) {
            w1[0][n] = wmm<C, K, true, false, LF, LF, true>(w1[0][n], XKs, U2s + 16 * t1.jt, &cs);
            bias(b1s, 16 * t1.jt, false);
          } else {
            w1[0][n] = wmm<C, K, true, false, LF, LF>(w1[0][n], XKs + 16 * t1.it, U2s + 16 * t1.jt);
          }
        }
      }
      take_next();
      put_w(s + 1, 0);
      stage_w1(0);
    }
    tgt = tgt_n;
    e_p = e_pn;
    e_s = e_sn;
  }
}

// One (chain, mini-batch): the readout up to Zb = Z2b without its bias (the
// Linear loop's Zb), in LDS; what the output and the backward need stays in
// LDS and registers.
template <typename T, class C> struct WideReadout {
  static constexpr int K = C::K, F = C::F, FF = C::FF, V = C::V, LS = C::LS, LF = C::LF, LK = C::LK, NSL = C::NSL,
                       NT = C::NT;
  using Sl = WideSlot<C>;
  typedef typename VecF<V>::type vf;
  static constexpr int LDS = 2 * C::SLOT + 7 * C::KSLOT;  // floats
  // LDS matrices (C1: -eta (A1 + 1), after forward() of the MLP -eta (A2 + 1);
  // Z: Z2b, in G1's place for the MLP)
  float *XQ, *XK, *G2, *W1, *W2, *X2, *XB, *C1, *Z;
  const float* slot;
  int w, prow, pcol;
  WideTile<4> ts;
  WideTile<C::FT> tf;
  WideTile<C::KT> tk;
  bool has_f, has_k;
  f4 eta, a1, a2;             // eta, XQ XK^T and X2b X2^T of the wave's K x K tile
  f4 xb[NSL], db[NSL];        // gelu(Z1b) and its derivative of its K x 64 tiles
  vf xq;                      // the thread's XQ row part

  __device__ __forceinline__ WideReadout(float* sm, const float* slot_)
      : slot(slot_), w(wide_wave<C>()), ts(w), tf(w), tk(w) {
    W1 = sm;
    W2 = sm + C::SLOT;
    sm += 2 * C::SLOT;
    XQ = sm;
    XK = sm + C::KSLOT;
    G2 = sm + 2 * C::KSLOT;
    X2 = sm + 3 * C::KSLOT;
    Z = sm + 4 * C::KSLOT;
    XB = sm + 5 * C::KSLOT;
    C1 = sm + 6 * C::KSLOT;
    prow = threadIdx.x >> 4;
    pcol = (threadIdx.x & 15) * V;
    has_f = C::f_tile(w);
    has_k = C::ALLK || w < C::KT * C::KT;
  }
  __device__ __forceinline__ void stage_w1(int sl) {
#pragma unroll
    for (int n = 0; n < NT; ++n) {
      const int t = w + n * C::NW;
      if (C::ALLT || t < C::TW) {
        const WideTile<4> t1(t);
        stf4(t1.template at<LS>(W1), ldf4(t1.template at<FF>(slot + Sl::W1 + sl * 64)));
      }
    }
  }
  __device__ __forceinline__ void stage_w2(int sl) {
#pragma unroll
    for (int n = 0; n < NT; ++n) {
      const int t = w + n * C::NW;
      if (C::ALLT || t < C::TW) {
        const WideTile<C::FT> t2(t);
        stf4(t2.template at<LF>(W2), ldf4(t2.template at<F>(slot + Sl::W2 + sl * 64 * F)));
      }
    }
  }
  // X2 = gelu(Z1) and G1 = P gelu'(Z1) of the wave's K x 64 tile
  __device__ __forceinline__ void inner(int sl, f4& x2, f4& g1) {
    const f4 z = ldf4(ts.template at<FF>(slot + Sl::Z1 + sl * 64)), p = ldf4(ts.template at<FF>(slot + Sl::P + sl * 64));
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      float y, dy;
      gelu_fwd_bwd(z[q], y, dy);
      x2[q] = y;
      g1[q] = p[q] * dy;
    }
  }
  __device__ __forceinline__ void stage_inner(int sl) {
    f4 x2, g1;
    inner(sl, x2, g1);
    stf4(ts.template at<LS>(X2), x2);
    stf4(ts.template at<LS>(Z), g1);
  }

  // ends with a barrier: Z is visible
  __device__ __forceinline__ void forward(const WideArgs& a, size_t m) {
    const unsigned po = (unsigned)(prow * F + pcol);
    xq = actf<T, V>(ldact<T, V>(static_cast<const T*>(a.XQ) + m * K * F + po));
    const vf xk = actf<T, V>(ldact<T, V>(static_cast<const T*>(a.XK) + m * K * F + po));
    const vf g2 = ldv<V>(slot + Sl::G2 + po);
    if (C::ALLK || has_k) eta = wide_eta4<T, K>(a, m, tk.row(), tk.col());
    stage_w1(0);
    if constexpr (C::MLP) {
      stage_w2(0);
      stage_inner(0);
    }
    stv<V>(XQ + prow * LF + pcol, xq);
    stv<V>(XK + prow * LF + pcol, xk);
    stv<V>(G2 + prow * LF + pcol, g2);
    __syncthreads();
    const f4 zero = f4{0.f, 0.f, 0.f, 0.f};
    if (C::ALLK || has_k) {
      a1 = wmm_on<WideFree<C>, F, false, true, LF, LF>(zero, XQ + 16 * tk.it * LF, XK + 16 * tk.jt * LF);
      stf4(tk.template at<LK>(C1), -(eta * (a1 + 1.0f)));
    }
    f4 z = zero;
    if constexpr (C::MLP) {
      a2 = zero;
#pragma unroll
      for (int sl = 0; sl < NSL; ++sl) {
        f4 zb = ldf4(slot + Sl::B1 + sl * 64 + ts.col());
        zb = wmm_on<WideFree<C>, F, false, false, LF, LS>(zb, XQ + 16 * ts.it * LF, W1 + 16 * ts.jt);
        if (sl == 0) __syncthreads();  // C1
        zb = wmm<WideFree<C>, K, false, false, LK, LS>(zb, C1 + 16 * ts.it * LK, Z + 16 * ts.jt);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          float y, dy;
          gelu_fwd_bwd(zb[q], y, dy);
          xb[sl][q] = y;
          db[sl][q] = dy;
        }
        stf4(ts.template at<LS>(XB), xb[sl]);
        __syncthreads();
        if (C::ALLK || has_k) a2 = wmm_sl<WideFree<C>, C::S, false, true, LS, LS>(a2, XB + 16 * tk.it * LS, X2 + 16 * tk.jt * LS);
        if (C::ALLF || has_f) z = wmm_sl<WideFree<C>, C::S, false, false, LS, LF>(z, XB + 16 * tf.it * LS, W2 + 16 * tf.jt);
        if (sl + 1 < NSL) {
          __syncthreads();
          stage_w1(sl + 1);
          stage_w2(sl + 1);
          stage_inner(sl + 1);
          __syncthreads();
        }
      }
      if (C::ALLK || has_k) stf4(tk.template at<LK>(C1), -(eta * (a2 + 1.0f)));
      __syncthreads();
      if (C::ALLF || has_f) {
        z = wmm<WideFree<C>, K, false, false, LK, LF>(z, C1 + 16 * tf.it * LK, G2 + 16 * tf.jt);
        stf4(tf.template at<LF>(Z), z);
      }
    } else {
      z = wmm_on<WideFree<C>, F, false, false, LF, LS>(z, XQ + 16 * tf.it * LF, W1 + 16 * tf.jt);
      __syncthreads();
      z = wmm<WideFree<C>, K, false, false, LK, LF>(z, C1 + 16 * tf.it * LK, G2 + 16 * tf.jt);
      stf4(tf.template at<LF>(Z), z);
    }
    __syncthreads();
  }
  // the normalised row part of Zb + bias
  __device__ __forceinline__ vf norm(float eps, float& sd) const {
    const vf z = ldv<V>(Z + prow * LF + pcol) + ldv<V>(slot + (C::MLP ? Sl::B2 : Sl::B1) + pcol);
    return wide_ln_row<V, F>(z, eps, sd);
  }
};

template <typename T, class C> __global__ __launch_bounds__(C::NTH) void wide_fwd_readout_kernel(WideArgs a) {
  constexpr int V = C::V;
  __shared__ __align__(16) float sm[WideReadout<T, C>::LDS];
  const size_t m = blockIdx.x;  // chain * NC + s
  const int h = (int)((m / (size_t)a.NC) % (size_t)a.H);
  WideReadout<T, C> ro(sm, a.saved + m * a.slot_stride);
  ro.forward(a, m);
  float sd;
  const typename VecF<V>::type xh = ro.norm(a.eps, sd);
  const float* lw = a.ln_w + (size_t)h * C::F + ro.pcol;
  const float* lb = a.ln_b + (size_t)h * C::F + ro.pcol;
  stact<T, V>(static_cast<T*>(a.out) + m * C::K * C::F + (unsigned)(ro.prow * C::F + ro.pcol),
              ro.xq + ldv<V>(lw) * xh + ldv<V>(lb));
}

}  // namespace
}  // namespace ttt
