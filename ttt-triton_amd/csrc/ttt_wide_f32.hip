// The ttt_wide.h kernels for fp32 activations.
#include "ttt_wide_inst.h"

namespace ttt {
template hipError_t launch_wide_t<float>(const WideArgs&, int, int, int, bool, bool, int, hipStream_t);
}  // namespace ttt
