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

// bytes of one (chain, mini-batch) slot, 0 for a shape that these kernels do not take
size_t wide_slot_bytes(int K, int F, int FF, bool mlp) {
  auto bytes = [](auto shape) { return WideSlot<decltype(shape)>::FLOATS * sizeof(float); };
  switch (K) {
    case 16: return wide_visit_kt<1>(F, FF, mlp, bytes);
    case 32: return wide_visit_kt<2>(F, FF, mlp, bytes);
    case 48: return wide_visit_kt<3>(F, FF, mlp, bytes);
    case 64: return wide_visit_kt<4>(F, FF, mlp, bytes);
    default: return 0;
  }
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
bool wide_shape_ok(int K, int F, int FF, bool mlp) { return K > 16 && wide_slot_bytes(K, F, FF, mlp) != 0; }

size_t wide_saved_bytes(int B, int H, int NC, int K, int F, int FF, bool mlp) {
  return (size_t)B * H * NC * wide_slot_bytes(K, F, FF, mlp);
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
  a.H = q.H;
  a.NC = q.NC;
  a.G = 1;
  a.M = 1;
  a.eta_rule = q.eta_rule;
  a.eps = q.eps;
  return launch_wide(a, q.B, q.K, q.F, q.FF, q.mlp, true, dtype, stream);
}

}  // namespace ttt
