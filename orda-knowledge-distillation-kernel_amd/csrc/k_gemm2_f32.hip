// k_gemm2_f32.hip -- general GEMM in fp32 for the exported orda_gemm where the
// split-operand engine has no layout: an MN-major A with a K-major B, and C of
// a column count off 4 (K-major operands).
#include "kernels.hpp"

namespace orda {
template <> hipError_t launch_gemm2<float>(const GemmParams& P, hipStream_t s) {
  using T = float;
  switch (P.la * 100 + P.lb * 10 + P.mode) {
    ORDA_GEMM2_CASE(KMAJ, KMAJ, GEMM_STORE)
    ORDA_GEMM2_CASE(MNMAJ, KMAJ, GEMM_STORE)
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}
}  // namespace orda
