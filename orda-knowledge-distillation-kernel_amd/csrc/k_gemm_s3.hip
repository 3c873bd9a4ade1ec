// k_gemm_s3.hip -- the fp32 gradient GEMMs (split-operand engine).
#include "split3.hpp"

namespace orda {

template <class C>
static hipError_t gemm_s3_go(const GemmParams& P, hipStream_t s) {
  const int64_t items = (int64_t)P.tiles_m * P.tiles_n * P.splits;
  if (items > 0x7fffffffll) return hipErrorInvalidValue;
  const int64_t resident = (int64_t)persistent_groups() * (C::MB == 4 ? 1 : 3);
  const dim3 g((unsigned)(items < resident ? items : resident)), b(C::kThreads);
  if (P.lb == KMAJ) {
    if (P.la != KMAJ || P.mode != GEMM_STORE || P.B1 || P.splits != 1) return hipErrorInvalidValue;
    hipLaunchKernelGGL((k_gemm_s3<C, KMAJ, KMAJ, GEMM_STORE>), g, b, 0, s, P);
  } else if (P.la == KMAJ && P.mode == GEMM_STORE) {
    hipLaunchKernelGGL((k_gemm_s3<C, KMAJ, MNMAJ, GEMM_STORE>), g, b, 0, s, P);
  } else if (P.la == KMAJ && P.mode == GEMM_ACC_T) {
    hipLaunchKernelGGL((k_gemm_s3<C, KMAJ, MNMAJ, GEMM_ACC_T>), g, b, 0, s, P);
  } else if (P.la == MNMAJ && P.mode == GEMM_STORE) {
    hipLaunchKernelGGL((k_gemm_s3<C, MNMAJ, MNMAJ, GEMM_STORE>), g, b, 0, s, P);
  } else if (P.la == MNMAJ && P.mode == GEMM_SPLIT) {
    hipLaunchKernelGGL((k_gemm_s3<C, MNMAJ, MNMAJ, GEMM_SPLIT>), g, b, 0, s, P);
  } else if (P.la == MNMAJ && P.mode == GEMM_ACC && P.splits == 1) {
    hipLaunchKernelGGL((k_gemm_s3<C, MNMAJ, MNMAJ, GEMM_ACC>), g, b, 0, s, P);
  } else {
    return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_gemm_s3(GemmParams P, hipStream_t s) {
  if (P.ldc % 4 != 0 || (P.lb == MNMAJ && P.N % 4 != 0) || P.splits < 1 || (P.B1 && P.splits != 1))
    return hipErrorInvalidValue;
  const bool big = s3_cost(P.M, P.N, P.K, P.splits, true) <= s3_cost(P.M, P.N, P.K, P.splits, false);
  auto tiles = [](int64_t n, int t) { return (int)((n + t - 1) / t); };
  P.tiles_m = tiles(P.M, big ? S3Big::kRowsA : S3Small::kRowsA);
  P.tiles_n = tiles(P.N, big ? S3Big::kRowsB : S3Small::kRowsB);
  return big ? gemm_s3_go<S3Big>(P, s) : gemm_s3_go<S3Small>(P, s);
}
}  // namespace orda
