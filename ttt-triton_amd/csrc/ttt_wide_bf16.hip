// The ttt_wide.h kernels for bf16 activations.
#include "ttt_wide_inst.h"

namespace ttt {
template hipError_t launch_wide_t<__bf16>(const WideArgs&, int, int, int, bool, bool, int, hipStream_t);
}  // namespace ttt
