// k_scan_f32.hip -- the fp32 scans (split-operand engine): losses and softmax
// statistics, without and with the logits store of the materialised path.
#include "split3.hpp"

namespace orda {

template <int SV, bool STORE>
static void scan_s3_go(const FusedParams& P, int grid, hipStream_t s) {
  if (P.tsrc == TSRC_SHARED) {
    hipLaunchKernelGGL((k_scan_s3<SV, STORE, S3_TIED>), dim3(grid), dim3(S3Big::kThreads), 0, s, P);
    return;
  }
  if constexpr (!STORE) {
    if (P.tsrc == TSRC_SEP) {
      hipLaunchKernelGGL((k_scan_s3<SV, STORE, S3_SEP>), dim3(grid), dim3(S3Big::kThreads), 0, s, P);
      return;
    }
  }
  hipLaunchKernelGGL((k_scan_s3<SV, STORE, S3_ALONE>), dim3(grid), dim3(S3Big::kThreads), 0, s, P);
}
// no teacher: student-only tiles
template <int SV, bool STORE>
static void scan_s3_alone(const FusedParams& P, int grid, hipStream_t s) {
  hipLaunchKernelGGL((k_scan_s3<SV, STORE, S3_ALONE>), dim3(grid), dim3(S3Big::kThreads), 0, s, P);
}
template <bool STORE>
static hipError_t scan_s3(const FusedParams& P, int grid, hipStream_t s) {
  if (P.tsrc == TSRC_MEM_RING || P.tsrc == (STORE ? TSRC_SEP : TSRC_L)) return hipErrorInvalidValue;
  switch (scan_variant_of(P)) {
    case SV_STUDENT: scan_s3_alone<SV_STUDENT, STORE>(P, grid, s); break;
    case SV_STUDENT_T: scan_s3_alone<SV_STUDENT_T, STORE>(P, grid, s); break;
    case SV_TCE_T1: scan_s3_go<SV_TCE_T1, STORE>(P, grid, s); break;
    case SV_TCE: scan_s3_go<SV_TCE, STORE>(P, grid, s); break;
    case SV_LIN_T1: scan_s3_go<SV_LIN_T1, STORE>(P, grid, s); break;
    case SV_LIN: scan_s3_go<SV_LIN, STORE>(P, grid, s); break;
    case SV_POW: scan_s3_go<SV_POW, STORE>(P, grid, s); break;
    case SV_POW1: scan_s3_go<SV_POW1, STORE>(P, grid, s); break;
    default:
      if constexpr (!STORE) {
        switch (scan_variant_of(P)) {
          case SV_JSD: scan_s3_go<SV_JSD, false>(P, grid, s); break;
          case SV_SKEW_F: scan_s3_go<SV_SKEW_F, false>(P, grid, s); break;
          case SV_SKEW_R: scan_s3_go<SV_SKEW_R, false>(P, grid, s); break;
          case SV_TVD: scan_s3_go<SV_TVD, false>(P, grid, s); break;
          default: return hipErrorInvalidValue;
        }
        break;
      }
      return hipErrorInvalidValue;
  }
  return hipGetLastError();
}
template <> hipError_t launch_scan<float>(const FusedParams& P, int grid, hipStream_t s) {
  return scan_s3<false>(P, grid, s);
}
template <> hipError_t launch_scan_store<float>(const FusedParams& P, int grid, hipStream_t s) {
  return P.phase != 0 ? hipErrorInvalidValue : scan_s3<true>(P, grid, s);
}
}  // namespace orda
