// The register-staged GEMM cores (operands at any element alignment, few-tile grids;
// gemm_kernels.h): their own translation unit, which builds beside k_gemm.hip.
#include "gemm_kernels.h"

namespace ghip {
template hipError_t launch_rs_tile<32, float, float>(GemmParams, hipStream_t);
template hipError_t launch_rs_tile<32, float, bf16_t>(GemmParams, hipStream_t);
template hipError_t launch_rs_tile<64, bf16_t, bf16_t>(GemmParams, hipStream_t);
template hipError_t launch_rs_tile<64, bf16_t, float>(GemmParams, hipStream_t);
template hipError_t launch_rs_tile<64, f16_t, f16_t>(GemmParams, hipStream_t);
template hipError_t launch_rs_tile<64, f16_t, float>(GemmParams, hipStream_t);
template hipError_t launch_rs_tile<64, float, float>(GemmParams, hipStream_t);
template hipError_t launch_rs_tile<64, float, bf16_t>(GemmParams, hipStream_t);
template hipError_t launch_rs_tile<128, bf16_t, bf16_t>(GemmParams, hipStream_t);
template hipError_t launch_rs_tile<128, bf16_t, float>(GemmParams, hipStream_t);
template hipError_t launch_rs_tile<128, f16_t, f16_t>(GemmParams, hipStream_t);
template hipError_t launch_rs_tile<128, f16_t, float>(GemmParams, hipStream_t);
template hipError_t launch_rs_tile<128, float, float>(GemmParams, hipStream_t);
template hipError_t launch_rs_tile<128, float, bf16_t>(GemmParams, hipStream_t);
}  // namespace ghip
