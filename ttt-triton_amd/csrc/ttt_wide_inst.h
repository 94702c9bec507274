// Launchers of the ttt_wide.h kernels for one activation type.
#pragma once

#include "ttt_wave16.h"
#include "ttt_wide_bwd.h"

namespace ttt {
namespace {

template <typename T, class C> hipError_t wide_fwd(const WideArgs& a, int chains, hipStream_t stream) {
  using Sl = WideSlot<C>;
  if constexpr (std::is_same_v<C, W16>) {
    if (a.slot_stride == Sl::FLOATS)
      hipLaunchKernelGGL((wave16_fwd_state_kernel<C, Sl::FLOATS>), dim3(chains), dim3(kW16Threads), 0, stream, a);
    else
      hipLaunchKernelGGL((wave16_fwd_state_kernel<C, Sl::FWD>), dim3(chains), dim3(kW16Threads), 0, stream, a);
  } else
    hipLaunchKernelGGL((wide_fwd_state_kernel<T, C>), dim3(chains), dim3(C::NTH), 0, stream, a);
  hipLaunchKernelGGL((wide_fwd_readout_kernel<T, C>), dim3(chains * a.NC), dim3(C::NTH), 0, stream, a);
  return hipGetLastError();
}
template <typename T, class C> hipError_t wide_bwd(const WideArgs& a, int chains, hipStream_t stream) {
  hipLaunchKernelGGL((wide_bwd_readout_kernel<T, C>), dim3(chains * a.NC), dim3(C::NTH), 0, stream, a);
  if constexpr (std::is_same_v<C, W16>)
    hipLaunchKernelGGL(wave16_bwd_state_kernel<C>, dim3(chains), dim3(kW16Threads), 0, stream, a);
  else
    hipLaunchKernelGGL((wide_bwd_state_kernel<T, C>), dim3(chains), dim3(C::NTH), 0, stream, a);
  return hipGetLastError();
}

template <typename T, int KT> hipError_t wide_kt(const WideArgs& a, int F, int FF, bool mlp, bool bwd, int chains,
                                                 hipStream_t stream) {
#define TTT_WIDE(FT, NSL, MLP)                                           \
  return bwd ? wide_bwd<T, WideShape<KT, FT, NSL, MLP>>(a, chains, stream) \
             : wide_fwd<T, WideShape<KT, FT, NSL, MLP>>(a, chains, stream)
  if (!mlp) TTT_WIDE(4, 1, false);
  if (F == 64 && FF == 64) TTT_WIDE(4, 1, true);
  if (F == 64 && FF == 256) TTT_WIDE(4, 4, true);
  if (F == 32 && FF == 128) TTT_WIDE(2, 2, true);
#undef TTT_WIDE
  return hipErrorInvalidValue;
}

}  // namespace

template <typename T>
hipError_t launch_wide_t(const WideArgs& a, int K, int F, int FF, bool mlp, bool bwd, int chains, hipStream_t stream) {
  switch (K) {
    case 16:
      if constexpr (sizeof(T) == 4) return wide_kt<T, 1>(a, F, FF, mlp, bwd, chains, stream);
      return hipErrorInvalidValue;
    case 32: return wide_kt<T, 2>(a, F, FF, mlp, bwd, chains, stream);
    case 48: return wide_kt<T, 3>(a, F, FF, mlp, bwd, chains, stream);
    case 64: return wide_kt<T, 4>(a, F, FF, mlp, bwd, chains, stream);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace ttt
