// The 256 x 128 GEMM core (gemm_kernels.h): its own translation unit, which builds
// beside k_gemm.hip.
#include "gemm_kernels.h"

namespace ghip {
template hipError_t launch_bf16_half<bf16_t, bf16_t>(GemmParams, bool, bool, hipStream_t);
template hipError_t launch_bf16_half<bf16_t, float>(GemmParams, bool, bool, hipStream_t);
template hipError_t launch_bf16_half<f16_t, f16_t>(GemmParams, bool, bool, hipStream_t);
template hipError_t launch_bf16_half<f16_t, float>(GemmParams, bool, bool, hipStream_t);
}  // namespace ghip
