#include "ols_gemm.h"

namespace tfcehip {

hipError_t launch_ols_gemm_bf16x3(const OlsGemmArgs& a, int tile, hipStream_t s) { return launch_split<2, false>(a, tile, s); }

}  // namespace tfcehip
