// TTT inner loops of mini-batches of 16 to 64 tokens on 64-wide heads (and
// of the 32-wide MLP with 128 hidden units): one workgroup holds a whole
// mini-batch in LDS and every product is 16 x 16 output tiles of fp32 MFMA,
// one K x 64 tile per wave.
//
// What bounds the shape is the recurrence: B*H chains, each NC mini-batches in
// a row, so a launch has B*H workgroups however long the sequence.  Only the
// products that the next mini-batch's state needs are therefore left in the
// per-chain launch; the readout, which reads a state and writes nothing that
// a later mini-batch reads, runs as a second launch with one workgroup per
// (chain, mini-batch), forward and backward alike:
//   wide_fwd_state    per chain: Z1, X2, Z2, G2, P = G2 W2^T, the update
//   wide_fwd_readout  per (chain, mini-batch): A1, Z1b, A2, Z2b, the output
//   wide_bwd_readout  per (chain, mini-batch): the readout again and its
//                     gradients: dXQ, most of deta, and what it adds to dG1,
//                     dG2, dX2, dXK, dW and db (the handoff)
//   wide_bwd_state    per chain, mini-batches in reverse: the update's gradient
// (the Linear loop has one layer: G, no P; the same four launches.)
//
// Measured at B32 H4, 8 mini-batches of 64 tokens, F = FF = 64, bf16, forward +
// backward: 429 us (MLP; state 77 + 172, readouts 53 + 132), where the
// general-shape kernels (one workgroup per chain for everything, every matrix
// through global scratch) take 6,780; the Linear loop 201 us against 3,090.
// The shapes taken are those that a layer (FF = F) or the 4x MLP builds of
// 32- and 64-wide heads; others keep the general-shape kernels.  64 chains of 8
// mini-batches, bf16, general-shape / these, us in a captured graph, forward and
// forward + backward (1 and 192 chains, 1 and 2 mini-batches and fp32 alike; none
// was slower here):
//           Linear 64            MLP 64/64             MLP 64/256               MLP 32/128
//   K = 32  385/38  1,379/99     815/67  2,906/190     2,838/191  10,199/922    889/77   3,176/228
//   K = 48  549/49  2,017/128  1,122/85  4,380/296     4,069/351  14,465/1,468  1,307/100  5,100/391
//   K = 64  719/55  2,685/149  1,478/99  5,934/314     5,530/361  19,796/1,597  1,805/118  6,915/446
//
// Mini-batches of 16 tokens in fp32 run here too where the caller asks for it
// (the split form, TTT_FORM_SPLIT): one wave per SIMD, so every product's operands
// are requested together and nothing waits behind a store.  Linear B2 H4, 16
// mini-batches, inference: 62 us in the specialised kernel, 36 here.
//
// Everything is held and summed in fp32 whatever the activation type, as in
// the general-shape kernels (ttt_generic.hip); activations are converted on
// load.  `saved` holds one slot per (chain, mini-batch), WideSlot below, with or
// without the handoff's place in it.
#pragma once

#include "ttt_eta.h"
#include "ttt_kernels.h"
#include "ttt_wide_layout.h"

namespace ttt {

struct WideArgs {
  const void *XQ, *XK, *XV, *eta, *dout;
  const float *ln_w, *ln_b;
  const float *W1_init, *b1_init, *W2_init, *b2_init;
  void* out;
  float *W1_last, *b1_last, *W2_last, *b2_last;
  float *W1_ckpt, *b1_ckpt, *W2_ckpt, *b2_ckpt;
  float *W1_memo, *b1_memo, *W2_memo, *b2_memo;
  void *dXQ, *dXK, *dXV, *deta;
  float *dW1, *db1, *dW2, *db2, *dln_w, *dln_b;
  float* saved;
  size_t slot_stride;   // (forward) floats from one slot to the next (backward: FLOATS)
  float* fin;           // (forward) where the state after a chain's last mini-batch goes
  size_t fin_stride;    // floats from one chain's to the next
  int H, NC, G, M, NI, eta_rule;
  float eps;
};

// The lane index, opaque once per use: what follows from it (some forty addresses)
// is then formed where it is used instead of being kept through a loop in registers
// that 16 waves do not have.
__device__ __forceinline__ int pinned(int l) {
  asm volatile("" : "+v"(l));
  return l & 63;  // (its range known again: 32-bit address offsets)
}
// The same for a slot's index: its addresses stay a scalar base and a lane offset.
__device__ __forceinline__ size_t pinned_index(size_t m) {
  asm volatile("" : "+s"(m));
  return m;
}

// ---------------------------------------------------------------- products
// c + op(A) op(B) for one 16 x 16 output tile, contraction KD (a multiple of
// 16): A and B point at the tile's first row (column) of op(A) (op(B)) in
// LDS.  op(A)[i][k] = TA ? A[k * LA + i] : A[i * LA + k], op(B)[k][j] = TB ?
// B[j * LB + k] : B[k * LB + j].  fp32 MFMA with the operands swapped, so that
// lane (g, r) holds C[r][4g .. 4g + 3]: four consecutive columns of one row
// (16-byte LDS and global accesses, per-row factors one scalar per lane).
// Of a single wave per SIMD (K = 16) every operand is requested before the first
// MFMA: left to itself the compiler waits for each pair of LDS reads in front of
// its two MFMAs.  (With four waves per SIMD the others' MFMAs cover that, and the
// batched reads queue: the MLP's state launches at K = F = FF = 64 took 10% more.)
// The product is summed by itself and added to c once: added to c term by term, a
// state took a rounding of its own size from each of the K terms of its update, and the
// gradients of K = 64 were 2.2 to 2.6 times as far from 64 bits as the general-shape
// kernels' (fp32, rms over five inputs: dXQ 2.6, dW1 2.2, out 2.2, now 1.0).  wmm_on
// starts from c instead: a term of the sum's own size (zero, a bias); wmm_sl adds the
// product of a hidden slice to the slices before it.  (The state launches of 16 tokens
// go on with c throughout: four MFMAs a term, errors below the specialised kernels'
// either way, and 8-10% less time.)
// With CS, `cs` receives op(B)'s column sums (column r, in every lane group).
// what may cross: VALU, SALU, VMEM, LDS writes; LDS reads and MFMAs may not
constexpr int kSchedKeepLdsReads = 0x2 | 0x4 | 0x70 | 0x200;
template <class C, int KD, bool TA, bool TB, int LA, int LB, bool CS = false, bool ON_ = false>
__device__ __forceinline__ f4 wmm(f4 c, const float* A, const float* B, float* cs = nullptr) {
  constexpr bool ON = ON_ || C::CHAIN;
  const int l = C::PIN ? pinned(lane_id()) : lane_id(), g = l >> 4, r = l & 15;
  const float* ap = TA ? A + 4 * g * LA + r : A + r * LA + 4 * g;
  const float* bp = TB ? B + r * LB + 4 * g : B + 4 * g * LB + r;
  Frag<float> a[KD / 16], b[KD / 16];
#pragma unroll
  for (int k = 0; k < KD; k += 16) {
    if constexpr (TA) {
#pragma unroll
      for (int j = 0; j < 4; ++j) a[k / 16].v[j] = ap[(k + j) * LA];
    } else {
      a[k / 16].v = *reinterpret_cast<const f4*>(ap + k);
    }
    if constexpr (TB) {
      b[k / 16].v = *reinterpret_cast<const f4*>(bp + k);
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j) b[k / 16].v[j] = bp[(k + j) * LB];
    }
  }
  if constexpr (C::KT == 1) __builtin_amdgcn_sched_barrier(kSchedKeepLdsReads);
  float t = 0.f;
  f4 p = ON ? c : f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int k = 0; k < KD / 16; ++k) {
    if constexpr (CS) t += (b[k].v[0] + b[k].v[1]) + (b[k].v[2] + b[k].v[3]);
    mma16(p, b[k], a[k]);
  }
  if constexpr (CS) *cs = sum_col4(t);
  if constexpr (ON) {
    return p;
  } else {
    // (c is taken up behind the product: brought forward it cost the FF = 256 backward 70
    // spilled registers of 128 more)
    asm volatile("" : "+v"(c[0]), "+v"(c[1]), "+v"(c[2]), "+v"(c[3]) : "v"(p[0]));
    return c + p;
  }
}

template <class C, int KD, bool TA, bool TB, int LA, int LB>
__device__ __forceinline__ f4 wmm_on(f4 c, const float* A, const float* B) {
  return wmm<C, KD, TA, TB, LA, LB, false, true>(c, A, B);
}

template <class C, int KD, bool TA, bool TB, int LA, int LB>
__device__ __forceinline__ f4 wmm_sl(f4 c, const float* A, const float* B) {
  return wmm<C, KD, TA, TB, LA, LB, false, (C::NSL == 1)>(c, A, B);
}

// this wave's index: uniform, below NW
template <class C> __device__ __forceinline__ int wide_wave() {
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  __builtin_assume(w >= 0 && w < C::NW);
  return w;
}

// the 16 x 16 tile grid of an R x Cc-tile product over the waves: tile w
template <int CT> struct WideTile {
  int it, jt, l;
  __device__ __forceinline__ explicit WideTile(int t, int lane = lane_id()) : it(t / CT), jt(t % CT), l(lane) {}
  __device__ __forceinline__ int row() const { return 16 * it + (l & 15); }
  __device__ __forceinline__ int col() const { return 16 * jt + 4 * (l >> 4); }
  // this lane's four columns in a matrix of row width LD: the tile's part of the
  // address is uniform over the wave, the lane's an unsigned offset (global
  // accesses then take a scalar base and one 32-bit register per row width)
  template <int LD, class P> __device__ __forceinline__ P* at(P* base) const {
    return base + (16 * it * LD + 16 * jt) + ((unsigned)(l & 15) * LD + 4u * (unsigned)(l >> 4));
  }
};

// ---------------------------------------------------------------- loads, stores
__device__ __forceinline__ f4 ldf4(const float* p) { return *reinterpret_cast<const f4*>(p); }
__device__ __forceinline__ void stf4(float* p, f4 v) { *reinterpret_cast<f4*>(p) = v; }

template <typename T> __device__ __forceinline__ Frag<T> ldraw4(const T* p) {
  Frag<T> f;
  f.v = *reinterpret_cast<const typename FragT<T>::type*>(p);
  return f;
}
template <typename T> __device__ __forceinline__ void st4(T* p, f4 v) {
  *reinterpret_cast<typename FragT<T>::type*>(p) = to_frag<T>(v).v;
}

// V = 2 or 4 consecutive values of a row pass
template <int V> struct VecF { typedef float type __attribute__((ext_vector_type(V))); };
template <typename T, int V> struct VecT { typedef T type __attribute__((ext_vector_type(V))); };
template <int V> __device__ __forceinline__ typename VecF<V>::type ldv(const float* p) {
  return *reinterpret_cast<const typename VecF<V>::type*>(p);
}
template <int V> __device__ __forceinline__ void stv(float* p, typename VecF<V>::type v) {
  *reinterpret_cast<typename VecF<V>::type*>(p) = v;
}
template <typename T, int V> __device__ __forceinline__ typename VecT<T, V>::type ldact(const T* p) {
  return *reinterpret_cast<const typename VecT<T, V>::type*>(p);
}
template <typename T, int V> __device__ __forceinline__ typename VecF<V>::type actf(typename VecT<T, V>::type x) {
  typename VecF<V>::type y;
#pragma unroll
  for (int q = 0; q < V; ++q) y[q] = (float)x[q];
  return y;
}
template <typename T, int V> __device__ __forceinline__ void stact(T* p, typename VecF<V>::type v) {
  f4 x = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int q = 0; q < V; ++q) x[q] = v[q];
  const Frag<T> f = to_frag<T>(x);
  typename VecT<T, V>::type y;
#pragma unroll
  for (int q = 0; q < V; ++q) y[q] = f.v[q];
  *reinterpret_cast<typename VecT<T, V>::type*>(p) = y;
}

// eta[K - 1][j] of a mini-batch whose eta (lr) starts at row0 = slot * K: as
// loaded, so that a request made ahead is not waited for where it is made ...
template <typename T, int K> __device__ __forceinline__ unsigned wide_eta_last_raw(const WideArgs& a, size_t slot, int j) {
  const size_t last = (slot * K + (K - 1)) * K + j;
  if constexpr (sizeof(T) == 2)
    if (a.eta_rule == TTT_ETA_DENSE) return static_cast<const unsigned short*>(a.eta)[last];
  const bool dense = a.eta_rule == TTT_ETA_DENSE || a.eta_rule == TTT_ETA_DENSE_F32;
  return static_cast<const unsigned*>(a.eta)[dense ? last : slot * K + j];
}
// ... and its value
template <typename T, int K> __device__ __forceinline__ float wide_eta_last_val(const WideArgs& a, unsigned raw) {
  if constexpr (sizeof(T) == 2)
    if (a.eta_rule == TTT_ETA_DENSE) return (float)__builtin_bit_cast(T, (unsigned short)raw);
  const float e = __builtin_bit_cast(float, raw);
  return a.eta_rule == TTT_ETA_LAYER || a.eta_rule == TTT_ETA_CAUSAL ? e * (1.0f / (float)K) : e;
}
// eta[i][j .. j + 3]
template <typename T, int K> __device__ __forceinline__ f4 wide_eta4(const WideArgs& a, size_t slot, int i, int j) {
  if (a.eta_rule == TTT_ETA_DENSE) return frag_to_f4(ldraw4(static_cast<const T*>(a.eta) + (slot * K + i) * K + j));
  const float* e = static_cast<const float*>(a.eta);
  if (a.eta_rule == TTT_ETA_DENSE_F32) return ldf4(e + (slot * K + i) * K + j);
  const f4 lr = ldf4(e + slot * K + j);
  if (a.eta_rule == TTT_ETA_LAYER) return lr * (1.0f / (float)K);
  const float c = 1.0f / (float)(i + 1);
  f4 r;
#pragma unroll
  for (int q = 0; q < 4; ++q) r[q] = j + q <= i ? lr[q] * c : 0.f;
  return r;
}
// coefficient of lr[j] in eta[i][j]
template <int K> __device__ __forceinline__ float wide_eta_coef(int rule, int i, int j) {
  if (rule == TTT_ETA_LAYER) return 1.0f / (float)K;
  return j <= i ? 1.0f / (float)(i + 1) : 0.f;
}

// ---------------------------------------------------------------- launchers
// one translation unit per activation type (ttt_wide_{f32,bf16,f16}.hip)
template <typename T>
hipError_t launch_wide_t(const WideArgs& a, int K, int F, int FF, bool mlp, bool bwd, int chains, hipStream_t stream);

}  // namespace ttt
