// Dispatch of the ttt_wide.h kernels: shapes, buffer size, launch.
#include "ttt_wide.h"

namespace ttt {

namespace {

// calls f(WideShape) for the shape's instantiation; 0 for any other shape
template <int KT, typename Fn> size_t wide_visit_kt(int F, int FF, bool mlp, Fn f) {
  if (!mlp) return F == 64 ? f(WideShape<KT, 4, 1, false>{}) : 0;
  if (F == 64 && FF == 64) return f(WideShape<KT, 4, 1, true>{});
  if (F == 64 && FF == 256) return f(WideShape<KT, 4, 4, true>{});
  if (F == 32 && FF == 128) return f(WideShape<KT, 2, 2, true>{});
  return 0;
}

template <typename Fn> size_t wide_visit(int K, int F, int FF, bool mlp, Fn f) {
  switch (K) {
    case 16: return wide_visit_kt<1>(F, FF, mlp, f);
    case 32: return wide_visit_kt<2>(F, FF, mlp, f);
    case 48: return wide_visit_kt<3>(F, FF, mlp, f);
    case 64: return wide_visit_kt<4>(F, FF, mlp, f);
    default: return 0;
  }
}

struct WideSizes {
  size_t fwd, floats, state, hst;  // of WideSlot; all 0 for a shape that these kernels do not take
};
WideSizes wide_sizes(int K, int F, int FF, bool mlp) {
  WideSizes z{};
  wide_visit(K, F, FF, mlp, [&z](auto s) {
    using Sl = WideSlot<decltype(s)>;
    z = {Sl::FWD, Sl::FLOATS, Sl::STATE, Sl::HST};
    return 1;
  });
  return z;
}

// Past this, mini-batches of 32 to 64 tokens take the general-shape kernels: a
// slot is 2 to 3 times the state that those keep of a mini-batch, and a training
// step holds every layer's until its backward.  (B32 H12 T2048 K64 F64 FF256: 3.4 GiB.)
constexpr size_t kWideMaxBytes = (size_t)4 << 30;

// One workgroup per slot: the forward's part of it to where the backward's
// launches read it.  Bound by its bytes: B16 H12, 32 mini-batches of 64, F 64, FF 256,
// 3.6 GB in 713 us, beside 6.8 ms of the backward's own launches.
__global__ __launch_bounds__(256) void wide_spread_kernel(const float* src, float* dst, int fwd, int floats) {
  src += (size_t)blockIdx.x * fwd;
  dst += (size_t)blockIdx.x * floats;
  for (int i = 4 * (int)threadIdx.x; i < fwd; i += 4 * 256) stf4(dst + i, ldf4(src + i));
}

hipError_t launch_wide(const WideArgs& a, int B, int K, int F, int FF, bool mlp, bool bwd, int dtype,
                       hipStream_t stream) {
  const int chains = B * a.H;
  if (dtype == TTT_DTYPE_BF16) return launch_wide_t<__bf16>(a, K, F, FF, mlp, bwd, chains, stream);
  if (dtype == TTT_DTYPE_F16) return launch_wide_t<_Float16>(a, K, F, FF, mlp, bwd, chains, stream);
  return launch_wide_t<float>(a, K, F, FF, mlp, bwd, chains, stream);
}

}  // namespace

// (16-token mini-batches only where the caller asks for the split form)
bool wide_runs(int B, int H, int NC, int K, int F, int FF, bool mlp) {
  const size_t slots = (size_t)B * H * NC * wide_sizes(K, F, FF, mlp).fwd * sizeof(float);
  return K > 16 && slots != 0 && slots <= kWideMaxBytes;
}

size_t wide_slots_bytes(int B, int H, int NC, int K, int F, int FF, bool mlp) {
  const WideSizes z = wide_sizes(K, F, FF, mlp);
  return (size_t)B * H * (NC * z.fwd + z.state) * sizeof(float);
}

size_t wide_saved_bytes(int B, int H, int NC, int K, int F, int FF, bool mlp) {
  return (size_t)B * H * NC * wide_sizes(K, F, FF, mlp).floats * sizeof(float);
}

hipError_t launch_wide_fwd(const GenFwdParams& q, int dtype, hipStream_t stream) {
  WideArgs a{};
  a.XQ = q.XQ;
  a.XK = q.XK;
  a.XV = q.XV;
  a.eta = q.eta;
  a.ln_w = q.ln_w;
  a.ln_b = q.ln_b;
  a.W1_init = q.W1_init;
  a.NI = q.NI;
  a.b1_init = q.b1_init;
  a.W2_init = q.W2_init;
  a.b2_init = q.b2_init;
  a.out = q.out;
  a.W1_last = q.W1_last;
  a.b1_last = q.b1_last;
  a.W2_last = q.W2_last;
  a.b2_last = q.b2_last;
  a.W1_ckpt = q.W1_ckpt;
  a.b1_ckpt = q.b1_ckpt;
  a.W2_ckpt = q.W2_ckpt;
  a.b2_ckpt = q.b2_ckpt;
  a.W1_memo = q.W1_memo;
  a.b1_memo = q.b1_memo;
  a.W2_memo = q.W2_memo;
  a.b2_memo = q.b2_memo;
  a.saved = static_cast<float*>(q.saved);
  const WideSizes z = wide_sizes(q.K, q.F, q.FF, q.mlp);
  if (q.slots) {  // the final states behind all slots
    a.slot_stride = z.fwd;
    a.fin = a.saved + (size_t)q.B * q.H * q.NC * z.fwd;
    a.fin_stride = z.state;
  } else {  // (in the last mini-batch's handoff, where the backward will write)
    a.slot_stride = z.floats;
    a.fin = a.saved + (q.NC - 1) * a.slot_stride + z.hst;
    a.fin_stride = q.NC * a.slot_stride;
  }
  a.H = q.H;
  a.NC = q.NC;
  a.G = q.G;
  a.M = q.M;
  a.eta_rule = q.eta_rule;
  a.eps = q.eps;
  return launch_wide(a, q.B, q.K, q.F, q.FF, q.mlp, false, dtype, stream);
}

hipError_t launch_wide_bwd(const GenBwdParams& q, int dtype, hipStream_t stream) {
  WideArgs a{};
  a.XQ = q.XQ;
  a.XK = q.XK;
  a.XV = q.XV;
  a.eta = q.eta;
  a.dout = q.dout;
  a.ln_w = q.ln_w;
  a.ln_b = q.ln_b;
  a.dXQ = q.dXQ;
  a.dXK = q.dXK;
  a.dXV = q.dXV;
  a.deta = q.deta;
  a.dW1 = q.dW1;
  a.db1 = q.db1;
  a.dW2 = q.dW2;
  a.db2 = q.db2;
  a.dln_w = q.dln_w;
  a.dln_b = q.dln_b;
  a.saved = static_cast<float*>(q.saved);
  if (q.spread != nullptr) {
    const WideSizes z = wide_sizes(q.K, q.F, q.FF, q.mlp);
    a.saved = static_cast<float*>(q.spread);
    hipLaunchKernelGGL(wide_spread_kernel, dim3(q.B * q.H * q.NC), dim3(256), 0, stream,
                       static_cast<const float*>(q.saved), a.saved, (int)z.fwd, (int)z.floats);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  a.H = q.H;
  a.NC = q.NC;
  a.G = 1;
  a.M = 1;
  a.eta_rule = q.eta_rule;
  a.eps = q.eps;
  return launch_wide(a, q.B, q.K, q.F, q.FF, q.mlp, true, dtype, stream);
}

}  // namespace ttt
