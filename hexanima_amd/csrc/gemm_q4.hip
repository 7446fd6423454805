// The GEMM kernels for int4 weights.
#define HXG_INSTANTIATE
#include "gemm_kernel.h"

namespace hxg {
HXG_LAUNCHES(, HXA_W_Q4, false)
HXG_LAUNCHES(, HXA_W_Q4, true)
}  // namespace hxg
