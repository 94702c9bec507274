// State launches of the split form (ttt_wide.h) for 16-token mini-batches of the
// 64-wide MLP with 256 hidden units, fp32: one workgroup of 16 waves per chain, wave
// w holds hidden units 16w .. 16w + 15: W1[:, its units] and W2[its units, :] (the
// backward: their gradients) as MFMA accumulators in registers for the whole
// sequence.  The slots in `saved` and the readout launches are ttt_wide.h's.
//
// What bounds it: fp32 MFMAs, 84 (forward) and 172 (backward) per wave and
// mini-batch at 32 cycles on four waves per SIMD, 4.5 and 9.2 us of the 8.9 and 19
// measured (B3 H5, 37 mini-batches), and the chain of two cross-wave row sums with
// the LayerNorm between them, where the matrix cores wait.  The specialised kernels,
// four waves carrying state and readout, take 14.6 and 24; hidden units in slices of
// 64 walked by four waves (ttt_wide.h) took 14 and 32.  16 waves leave 128 registers
// each: addresses are kept out of them (pinned, pinned_index below: 977 -> 703 us for
// the backward, whose spills waited behind its loads).
//
// Layouts, for 16 x 16 blocks and lane (g, n) = (lane / 16, lane % 16), registers j:
//   "T"  [unit 4g + j][token n]     elementwise values of the hidden layer
//   "C"  [token 4g + j][unit n]     the same transposed (one exact MFMA pass each)
// An accumulator [rows 4g + j][cols n] is an operand whose free index is its column
// and whose contraction index is its row, so T feeds products over units, C products
// over tokens, W1 and dW1 [feature][unit] and dW2^T [feature][unit] products over
// features.  What contracts the other way comes from LDS or from global rows.
#pragma once

#include "ttt_wide.h"

namespace ttt {
namespace {

using W16 = WideShape<1, 4, 4, true>;
constexpr int kW16Waves = 16, kW16Threads = 64 * kW16Waves;
constexpr int kRowLd = 68;  // [16][64] rows in LDS: 16-byte row reads and 4-byte column reads without bank conflicts
constexpr int kColLd = 20;  // [64][16] columns in LDS

__device__ __forceinline__ Frag<float> fr(f4 v) { return Frag<float>{v}; }
// 16-byte row read of an operand: free index r = lane % 16, contraction 4g + j
template <int LD> __device__ __forceinline__ Frag<float> row_frag(const float* m, int l) {
  return fr(ldf4(m + (l & 15) * LD + 4 * (l >> 4)));
}
// column read: free index lane % 16 along a row, contraction over rows 4g + j
__device__ __forceinline__ Frag<float> col_frag(const float* m, int ld, int l) {
  f4 v;
#pragma unroll
  for (int j = 0; j < 4; ++j) v[j] = m[(unsigned)((4 * (l >> 4) + j) * ld + (l & 15))];
  return fr(v);
}
__device__ __forceinline__ f4 w16_flip(f4 v, int l) {  // T <-> C
  f4 ident;
#pragma unroll
  for (int j = 0; j < 4; ++j) ident[j] = 4 * (l >> 4) + j == (l & 15) ? 1.0f : 0.0f;
  return transpose16(fr(v), fr(ident)).v;
}

// sum over the waves of part[wave][row][lane]
__device__ __forceinline__ float wave_parts(const float* part, int row, int l) {
  float s[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int p = 0; p < kW16Waves; ++p) s[p & 3] += part[(p * 16 + row) * kRowLd + l];
  return (s[0] + s[1]) + (s[2] + s[3]);
}

// eta's last row of slot m: token n's value, raw (see wide_eta_last_raw)
__device__ __forceinline__ unsigned w16_eta(const WideArgs& a, size_t m, int tok) {
  return wide_eta_last_raw<float, 16>(a, m, tok);
}

// (templates: compiled where they are launched, in the fp32 translation unit)
// STRIDE: floats from one slot to the next (from the arguments: 325 -> 333 us at B3 H5, 37 mini-batches)
template <class C, int STRIDE> __global__ __launch_bounds__(kW16Threads) void wave16_fwd_state_kernel(WideArgs a) {
  constexpr int K = 16, F = 64, FF = 256;
  using Sl = WideSlot<C>;
  __shared__ __align__(16) float part[kW16Waves][16][kRowLd];  // a wave's W2 rows, then its share of Z2
  __shared__ __align__(16) float xk[2][16][kRowLd], xkT[2][F][kColLd];
  __shared__ __align__(16) float g2[16][kRowLd], u2T[F][kColLd];
  __shared__ __align__(16) float b1s[FF], b2s[F];
  const size_t chain = blockIdx.x;
  const int h = (int)(chain % (size_t)a.H), NC = a.NC;
  const int tid = threadIdx.x, l = tid & 63, g = l >> 4, n = l & 15;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int NK = (NC + a.G - 1) / a.G, NS = (NC + a.M - 1) / a.M;
  float* const slot0 = a.saved + chain * NC * (size_t)STRIDE;
  const float lw = a.ln_w[(size_t)h * F + l], lb = a.ln_b[(size_t)h * F + l];
  float* const own = &part[w][0][0];

  // W1[i]: [feature 16i + 4g + j][unit n], W2[c]: [unit 4g + j][feature 16c + n]
  f4 W1[4], W2[4];
  const size_t ic = chain % (size_t)a.NI;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    W1[i] = col_frag(a.W1_init + ic * F * FF + 16 * i * FF + 16 * w, FF, l).v;
    W2[i] = col_frag(a.W2_init + (ic * FF + 16 * w) * F + 16 * i, F, l).v;
  }
  if (tid < FF) b1s[tid] = a.b1_init[ic * FF + tid];
  if (tid < F) b2s[tid] = a.b2_init[ic * F + tid];
  auto rows_to_lds = [&]() {  // W2's rows, for the products over features
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
      for (int j = 0; j < 4; ++j) own[(4 * g + j) * kRowLd + 16 * c + n] = W2[c][j];
  };
  rows_to_lds();

  // the state (b1 and b2 included) to one destination
  f4 w2r[4];  // [unit n][feature 16c + 4g + j]
  auto put = [&](float* pW1, float* pb1, float* pW2, float* pb2) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
      for (int j = 0; j < 4; ++j) (pW1 + (16 * i + j) * FF + 16 * w)[(unsigned)(4 * g * FF + n)] = W1[i][j];
      stf4(pW2 + 16 * w * F + 16 * i + (unsigned)(n * F + 4 * g), w2r[i]);
    }
    if (l < 16 && pb1 != nullptr) (pb1 + 16 * w)[(unsigned)l] = b1s[16 * w + l];
    if (w == 15 && pb2 != nullptr) pb2[(unsigned)l] = b2s[l];
  };
  // checkpoints and snapshots are counted, not divided for
  int ck = 0, ck_in = 0, mk = 0, mk_in = 1;
  auto emit = [&](int s) {  // the state entering mini-batch s
    if (s < NC) {
      float* q = slot0 + (size_t)s * STRIDE;
      put(q + Sl::W1, q + Sl::B1, q + Sl::W2, q + Sl::B2);
      if (ck_in == 0 && a.W1_ckpt != nullptr) {
        // (only W1's checkpoints are always there)
        const size_t k = chain * NK + ck;
        float* const none = nullptr;
        if (a.W2_ckpt != nullptr)
          put(a.W1_ckpt + k * F * FF, a.b1_ckpt ? a.b1_ckpt + k * FF : none, a.W2_ckpt + k * FF * F,
              a.b2_ckpt ? a.b2_ckpt + k * F : none);
        else
#pragma unroll
          for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j)
              (a.W1_ckpt + k * F * FF + (16 * i + j) * FF + 16 * w)[(unsigned)(4 * g * FF + n)] = W1[i][j];
        if (a.W2_ckpt == nullptr) {
          if (l < 16 && a.b1_ckpt != nullptr) (a.b1_ckpt + k * FF + 16 * w)[(unsigned)l] = b1s[16 * w + l];
          if (w == 15 && a.b2_ckpt != nullptr) (a.b2_ckpt + k * F)[(unsigned)l] = b2s[l];
        }
      }
    } else if (a.W1_last != nullptr) {
      put(a.W1_last + chain * F * FF, a.b1_last + chain * FF, a.W2_last + chain * FF * F, a.b2_last + chain * F);
    }
    if (mk_in == 0 && a.W1_memo != nullptr) {
      const size_t k = chain * NS + mk;
      put(a.W1_memo + k * F * FF, a.b1_memo + k * FF, a.W2_memo + k * FF * F, a.b2_memo + k * F);
    }
    if (--ck_in < 0) {
      ck_in = a.G - 1;
      ++ck;
    }
    if (--mk_in < 0) {
      mk_in = a.M - 1;
      ++mk;
    }
  };

  const float* const XK = static_cast<const float*>(a.XK);
  const float* const XV = static_cast<const float*>(a.XV);
  float x = (XK + chain * NC * K * F)[(unsigned)tid], tgt = (XV + chain * NC * K * F)[(unsigned)tid] - x;  // token w, feature l
  float xn = 0.f, vn = 0.f;
  unsigned er = w16_eta(a, chain * NC, w), en[4];
  auto eta_tokens = [&](size_t m) {  // tokens 4g + j
#pragma unroll
    for (int j = 0; j < 4; ++j) en[j] = w16_eta(a, m, 4 * g + j);
  };
  eta_tokens(chain * NC);
  xk[0][w][l] = x;
  xkT[0][l][w] = x;
  __syncthreads();

  for (int s = 0; s < NC; ++s) {
    const int l = pinned(lane_id()), g = l >> 4, n = l & 15, tid = 64 * w + l;
    const int b = s & 1;
    const size_t m = pinned_index(chain * NC + s);
    float* const slot = a.saved + m * STRIDE;
    float e_r = wide_eta_last_val<float, K>(a, er);
    f4 e4;
#pragma unroll
    for (int j = 0; j < 4; ++j) e4[j] = wide_eta_last_val<float, K>(a, en[j]);
    f4 z = ldf4(b1s + 16 * w + 4 * g);
#pragma unroll
    for (int c = 0; c < 4; ++c) w2r[c] = row_frag<kRowLd>(own + 16 * c, l).v;
    {  // Z1 in T: W1^T XK^T + b1
      Frag<float> q[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) q[i] = row_frag<kRowLd>(&xk[b][0][16 * i], l);
#pragma unroll
      for (int i = 0; i < 4; ++i) mma16(z, fr(W1[i]), q[i]);
    }
    f4 x2t;
#pragma unroll
    for (int j = 0; j < 4; ++j) x2t[j] = gelu_tanh(z[j]);
#pragma unroll
    for (int c = 0; c < 4; ++c) {  // this wave's share of Z2^T, [feature 16c + 4g + j][token n]
      f4 p = f4{0.f, 0.f, 0.f, 0.f};
      mma16(p, fr(W2[c]), fr(x2t));
      stf4(own + n * kRowLd + 16 * c + 4 * g, p);
    }
    emit(s);
    stf4(slot + Sl::Z1 + 16 * w + (unsigned)(n * FF + 4 * g), z);
    if (s + 1 < NC) {
      xn = (XK + (m + 1) * K * F)[(unsigned)tid];
      vn = (XV + (m + 1) * K * F)[(unsigned)tid];
      er = w16_eta(a, m + 1, w);
      eta_tokens(m + 1);
    }
    const f4 zc = w16_flip(z, l);
    f4 x2, d1;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      float y, dy;
      gelu_fwd_bwd(zc[j], y, dy);
      x2[j] = y;
      d1[j] = dy;
    }
    __syncthreads();
    {  // token w: LayerNorm fused with the L2 loss's gradient
      float v = b2s[l] + wave_parts(&part[0][0][0], w, l);
      v -= sum_wave(v) * (1.0f / F);
      const float sd = sqrtf(sum_wave(v * v) * (1.0f / F) + a.eps);
      const float rs = 1.0f / sd, xh = v * rs;
      float gr = lw * (lw * xh + lb - tgt);
      const float s1 = sum_wave(gr) * (1.0f / F), s2 = sum_wave(gr * xh) * (1.0f / F);
      gr = (gr - s1 - xh * s2) * rs;
      g2[w][l] = gr;
      u2T[l][w] = gr * -e_r;
      (slot + Sl::G2)[(unsigned)tid] = gr;
      (slot + Sl::ZH)[(unsigned)tid] = xh;
      if (l == 0) slot[Sl::SIG + w] = sd;
      if (s + 1 < NC) {  // the next mini-batch's rows, into the other buffer
        x = xn;
        tgt = vn - xn;
        xk[b ^ 1][w][l] = x;
        xkT[b ^ 1][l][w] = x;
      }
    }
    __syncthreads();
    f4 p = f4{0.f, 0.f, 0.f, 0.f};  // P = G2 W2^T in C
    {
      Frag<float> q[4];
#pragma unroll
      for (int c = 0; c < 4; ++c) q[c] = row_frag<kRowLd>(&g2[0][16 * c], l);
#pragma unroll
      for (int c = 0; c < 4; ++c) mma16(p, q[c], fr(w2r[c]));
    }
    const f4 u1 = p * d1 * -e4;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      mma16(W2[i], fr(x2), row_frag<kColLd>(&u2T[16 * i][0], l));
      mma16(W1[i], row_frag<kColLd>(&xkT[b][16 * i][0], l), fr(u1));
    }
    rows_to_lds();
#pragma unroll
    for (int j = 0; j < 4; ++j) (slot + Sl::P + j * FF + 16 * w)[(unsigned)(4 * g * FF + n)] = p[j];
    const float bs = sum_col4((u1[0] + u1[1]) + (u1[2] + u1[3]));
    if (l < 16) b1s[16 * w + l] += bs;
    if (w == 15) {
      f4 t = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int q = 0; q < 4; ++q) t += ldf4(&u2T[l][4 * q]);
      b2s[l] += (t[0] + t[1]) + (t[2] + t[3]);
    }
  }
#pragma unroll
  for (int c = 0; c < 4; ++c) w2r[c] = row_frag<kRowLd>(own + 16 * c, l).v;
  emit(NC);
}

// Per chain, the mini-batches in reverse: the gradient through the update (see
// wide_bwd_state_kernel), carrying dW1 [feature 16i + 4g + j][unit n] and dW2^T
// [feature 16c + 4g + j][unit n].  Their products over units take operands that
// pass through the wave's own rows in LDS.
template <class C> __global__ __launch_bounds__(kW16Threads) void wave16_bwd_state_kernel(WideArgs a) {
  constexpr int K = 16, F = 64, FF = 256;
  using Sl = WideSlot<C>;
  __shared__ __align__(16) float part[kW16Waves][16][kRowLd];
  __shared__ __align__(16) float xk[16][kRowLd], g2[16][kRowLd], dz2[16][kRowLd];
  __shared__ __align__(16) float xkT[F][kColLd], g2T[F][kColLd], dz2T[F][kColLd];
  __shared__ __align__(16) float db1s[FF], db2s[F], dep[kW16Waves + 1][K];
  const size_t chain = blockIdx.x;
  const int h = (int)(chain % (size_t)a.H), NC = a.NC;
  const int tid = threadIdx.x, l = tid & 63, g = l >> 4, n = l & 15;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  float* const slot0 = a.saved + chain * NC * (size_t)Sl::FLOATS;
  const float lw = a.ln_w[(size_t)h * F + l], lb = a.ln_b[(size_t)h * F + l];
  float* const own = &part[w][0][0];
  const f4 zero = f4{0.f, 0.f, 0.f, 0.f};
  f4 dW1[4], dW2t[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) dW1[i] = dW2t[i] = zero;
  if (tid < FF) db1s[tid] = 0.f;
  if (tid < F) db2s[tid] = 0.f;
  float accw = 0.f, accb = 0.f, hln = 0.f;
  const float* const XK = static_cast<const float*>(a.XK);
  const float* const XV = static_cast<const float*>(a.XV);
  // token w, feature l of a mini-batch
  size_t m = chain * NC + NC - 1;
  float xw = (XK + m * K * F)[(unsigned)tid], gw = (slot0 + (size_t)(NC - 1) * Sl::FLOATS + Sl::G2)[(unsigned)tid];
  auto stage_rows = [&]() {
    xk[w][l] = xw;
    xkT[l][w] = xw;
    g2[w][l] = gw;
    g2T[l][w] = gw;
  };
  stage_rows();
  __syncthreads();

  for (int s = NC - 1; s >= 0; --s) {
    const int l = pinned(lane_id()), g = l >> 4, n = l & 15, tid = 64 * w + l;
    m = pinned_index(chain * NC + s);
    float* const slot = a.saved + m * Sl::FLOATS;
    auto ldT = [&](int off) { return ldf4(slot + off + 16 * w + (unsigned)(n * FF + 4 * g)); };
    const f4 z = ldT(Sl::Z1), p = ldT(Sl::P), hg1 = ldT(Sl::HG1), hx2 = ldT(Sl::HX2);
    const unsigned en = w16_eta(a, m, n), er = w16_eta(a, m, w);
    if (w < 2) hln += (slot + Sl::HLW)[(unsigned)tid];  // (HLB follows HLW)
    const float e = wide_eta_last_val<float, K>(a, en);
    // ---- through the update: t1 = XK dW1 + db1, q2 = G2 dW2^T, both T
    f4 t1 = ldf4(db1s + 16 * w + 4 * g), q2 = zero;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      mma16(t1, fr(dW1[i]), row_frag<kRowLd>(&xk[0][16 * i], l));
      mma16(q2, fr(dW2t[i]), row_frag<kRowLd>(&g2[0][16 * i], l));
    }
    f4 x2, d1, dd1;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      float y, dy, ddy;
      gelu_all(z[j], y, dy, ddy);
      x2[j] = y;
      d1[j] = dy;
      dd1[j] = ddy;
    }
    const f4 g1 = p * d1;
    {
      const f4 de = t1 * g1 + x2 * q2;
      const float d = sum_col4((de[0] + de[1]) + (de[2] + de[3]));
      if (l < 16) dep[w][l] = -d;
    }
    const f4 dg1 = hg1 - t1 * e;
    const f4 dz1a = dg1 * p * dd1, dp = dg1 * d1, dx2 = hx2 - q2 * e;
    const f4 ng1 = g1 * -e;
    {  // dG2 - t2 e, [feature 16c + 4g + j][token n]: dW2 over units, through this wave's rows [unit][feature]
      f4 dg[4];
      const f4 nx2 = x2 * -e;
#pragma unroll
      for (int c = 0; c < 4; ++c) stf4(own + n * kRowLd + 16 * c + 4 * g, dW2t[c]);
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        dg[c] = zero;
        mma16(dg[c], col_frag(slot + Sl::W2 + 16 * w * F + 16 * c, F, l), fr(dp));
        mma16(dg[c], col_frag(own + 16 * c, kRowLd, l), fr(nx2));
      }
#pragma unroll
      for (int c = 0; c < 4; ++c) stf4(own + n * kRowLd + 16 * c + 4 * g, dg[c]);
    }
    const f4 x2c = w16_flip(x2, l), dpc = w16_flip(dp, l);
    const float xv = (XV + m * K * F)[(unsigned)tid], zh = (slot + Sl::ZH)[(unsigned)tid];
    const float hg2 = (slot + Sl::HG2)[(unsigned)tid], sd = slot[Sl::SIG + w];
    f4 w2r[4];  // [unit n][feature 4g + j], requested in front of the LayerNorm phase, used behind it
#pragma unroll
    for (int i = 0; i < 4; ++i) w2r[i] = ldf4(slot + Sl::W2 + 16 * w * F + 16 * i + (unsigned)(n * F + 4 * g));
    if (s > 0) {
      xw = (XK + (m - 1) * K * F)[(unsigned)tid];
      gw = (slot - Sl::FLOATS + Sl::G2)[(unsigned)tid];
    }
    __syncthreads();
    float dt;
    {  // token w: backward of the LayerNorm fused with the L2 loss's gradient
      const float e_r = wide_eta_last_val<float, K>(a, er), rs = 1.0f / sd, inv = rs * (1.0f / F);
      const float db2 = db2s[l], xcur = xk[w][l], gcur = g2[w][l];
      const float qv = wave_parts(&part[0][0][0], w, l) + hg2 - e_r * db2;
      const float rr = lw * zh + lb - (xv - xcur), gx = lw * rr;
      const f4 sums = sum4_wave(f4{gx * zh, qv, qv * zh, qv * gcur});
      const float S2 = sums[0], Q1 = sums[1], Q2 = sums[2], QG = sums[3];
      const float dgr = ((float)F * qv - Q1 - zh * Q2) * inv;
      dt = -(dgr * lw);
      accw += dgr * (rr + lw * zh);
      accb += dgr * lw;
      const float dxh = (-qv * S2 - gx * Q2) * inv + dgr * lw * lw;
      const f4 ms = sum4_wave(f4{dxh, dxh * zh, db2 * gcur, 0.f});
      const float dz = (dxh - ms[0] * (1.0f / F) - zh * (ms[1] * (1.0f / F))) * rs - zh * (QG * rs * (1.0f / F));
      if (l == 0) dep[kW16Waves][w] = -ms[2];
      dz2[w][l] = dz;
      dz2T[l][w] = dz;
      (static_cast<float*>(a.dXV) + m * K * F)[(unsigned)tid] = dt;
    }
    __syncthreads();
    if (w == 0 && l < K) {  // deta's last row (dlr): the readout's terms and the update's
      float d = 0.f;
#pragma unroll
      for (int q = 0; q <= kW16Waves; ++q) d += dep[q][tid];
      const float hd = (slot + Sl::HDE)[(unsigned)tid];
      if (a.eta_rule == TTT_ETA_DENSE || a.eta_rule == TTT_ETA_DENSE_F32)
        (static_cast<float*>(a.deta) + (m * K + (K - 1)) * K)[(unsigned)tid] = hd + d;
      else
        (static_cast<float*>(a.deta) + m * K)[(unsigned)tid] = hd + d * (1.0f / (float)K);
    }
    f4 w1r[4];  // [feature n][unit 4g + j]
#pragma unroll
    for (int i = 0; i < 4; ++i) w1r[i] = ldf4(slot + Sl::W1 + 16 * i * FF + 16 * w + (unsigned)(n * FF + 4 * g));
    f4 dx = dx2;  // + dZ2 W2^T
#pragma unroll
    for (int c = 0; c < 4; ++c)
      mma16(dx, fr(w2r[c]), row_frag<kRowLd>(&dz2[0][16 * c], l));
    const f4 dz1 = dz1a + dx * d1;
    {  // dXK, [feature 16i + 4g + j][token n]: dW1 over units the same way (the waves' shares of dZ2
       // were all read before the last barrier)
      f4 dxk[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) stf4(own + n * kRowLd + 16 * i + 4 * g, dW1[i]);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        dxk[i] = zero;
        mma16(dxk[i], col_frag(own + 16 * i, kRowLd, l), fr(ng1));
        mma16(dxk[i], fr(w1r[i]), fr(dz1));
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) stf4(own + n * kRowLd + 16 * i + 4 * g, dxk[i]);
    }
    const f4 dz1c = w16_flip(dz1, l);
    const float hxk = (slot + Sl::HXK)[(unsigned)tid];
    f4 h1[4], h2[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      h2[i] = ldf4(slot + Sl::HST + Sl::W2 + 16 * w * F + 16 * i + (unsigned)(n * F + 4 * g));
      h1[i] = col_frag(slot + Sl::HST + Sl::W1 + 16 * i * FF + 16 * w, FF, l).v;
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      mma16(dW2t[i], row_frag<kColLd>(&g2T[16 * i][0], l), fr(dpc));
      mma16(dW2t[i], row_frag<kColLd>(&dz2T[16 * i][0], l), fr(x2c));
      mma16(dW1[i], row_frag<kColLd>(&xkT[16 * i][0], l), fr(dz1c));
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      dW2t[i] += h2[i];
      dW1[i] += h1[i];
    }
    const float bs = sum_col4((dz1c[0] + dz1c[1]) + (dz1c[2] + dz1c[3]));
    if (l < 16) db1s[16 * w + l] += bs + (slot + Sl::HST + Sl::B1 + 16 * w)[(unsigned)l];
    if (w == 15) {
      f4 t = zero;
#pragma unroll
      for (int q = 0; q < 4; ++q) t += ldf4(&dz2T[l][4 * q]);
      db2s[l] += ((t[0] + t[1]) + (t[2] + t[3])) + (slot + Sl::HST + Sl::B2)[(unsigned)l];
    }
    __syncthreads();
    (static_cast<float*>(a.dXK) + m * K * F)[(unsigned)tid] = wave_parts(&part[0][0][0], w, l) + hxk - dt;
    stage_rows();
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
#pragma unroll
    for (int j = 0; j < 4; ++j)
      (a.dW1 + chain * F * FF + (16 * i + j) * FF + 16 * w)[(unsigned)(4 * g * FF + n)] = dW1[i][j];
    stf4(a.dW2 + (chain * FF + 16 * w) * F + 16 * i + (unsigned)(n * F + 4 * g), dW2t[i]);
  }
  if (tid < FF) a.db1[chain * FF + tid] = db1s[tid];
  if (tid < F) a.db2[chain * F + tid] = db2s[tid];
  own[l] = accw;
  own[kRowLd + l] = accb;
  __syncthreads();
  if (tid < 2 * F) {  // wave 0: dln_w, wave 1: dln_b
    float t = hln;
#pragma unroll
    for (int q = 0; q < kW16Waves; ++q) t += part[q][w][l];
    (w == 0 ? a.dln_w : a.dln_b)[chain * F + l] = t;
  }
}

}  // namespace
}  // namespace ttt
