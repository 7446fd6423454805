// The GEMM kernels for fp16 weights.
#define HXG_INSTANTIATE
#include "gemm_kernel.h"

namespace hxg {
HXG_LAUNCHES(, HXA_W_F16, false)

// the cross-q projection with its attention (xattn_tail): 128 x 128 fp16 tiles, 4 waves
__global__ __launch_bounds__(256, 2) void gemm_xattn_kernel(GemmParams p) {
  gemm_body<128, 128, HXA_W_F16, false, false, 4, true>(p, blockIdx.x, 0);
}
hipError_t launch_xattn(const GemmParams &p, hipStream_t st) {
  constexpr int lds = XA_LDS;
  static bool attr = false;
  if (!attr) {
    const hipError_t e = hipFuncSetAttribute((const void *)gemm_xattn_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (e != hipSuccess) return e;
    attr = true;
  }
  hxa_launch(gemm_xattn_kernel, dim3(p.tiles_m * p.tiles_n), dim3(256), lds, st, p);
  return hipGetLastError();
}
}  // namespace hxg
