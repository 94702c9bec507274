// The ttt_wide.h kernels for fp16 activations.
#include "ttt_wide_inst.h"

namespace ttt {
template hipError_t launch_wide_t<_Float16>(const WideArgs&, int, int, int, bool, bool, int, hipStream_t);
}  // namespace ttt
