#include "ols_gemm.h"

namespace tfcehip {

hipError_t launch_ols_gemm_fp32(const OlsGemmArgs& a, hipStream_t s) {
  const dim3 grid(gemm_blocks(a)), block(256);
  switch (epi_kind(a)) {
    case kEpiT1: hipLaunchKernelGGL(ols_gemm_fp32_kernel<kEpiT1>, grid, block, 0, s, a); break;
    case kEpiT2: hipLaunchKernelGGL(ols_gemm_fp32_kernel<kEpiT2>, grid, block, 0, s, a); break;
    case kEpiT4: hipLaunchKernelGGL(ols_gemm_fp32_kernel<kEpiT4>, grid, block, 0, s, a); break;
    case kEpiT7: hipLaunchKernelGGL(ols_gemm_fp32_kernel<kEpiT7>, grid, block, 0, s, a); break;
    case kEpiPair: hipLaunchKernelGGL(ols_gemm_fp32_kernel<kEpiPair>, grid, block, 0, s, a); break;
    case kEpiF: hipLaunchKernelGGL(ols_gemm_fp32_kernel<kEpiF>, grid, block, 0, s, a); break;
    case kEpiBlk: hipLaunchKernelGGL(ols_gemm_fp32_kernel<kEpiBlk>, grid, block, 0, s, a); break;
  }
  return hipGetLastError();
}

}  // namespace tfcehip
