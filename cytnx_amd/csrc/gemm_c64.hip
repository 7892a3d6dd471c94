// Grouped GEMM launches in complex64.
#define CXA_GEMM_TU c64
#include "gemm_kernels.hpp"

namespace cxa {

int launch_gemm_c64(const GemmLaunch &g, hipStream_t s) {
  return launch_t<CXA_PREC_FP32, cf, cf, cf, true>(g, s);
}

}  // namespace cxa
