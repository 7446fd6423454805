// The GEMM kernels for int8 weights.
#define HXG_INSTANTIATE
#include "gemm_kernel.h"

namespace hxg {
HXG_LAUNCHES(, HXA_W_Q8, false)
}  // namespace hxg
