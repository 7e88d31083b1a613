// Backward kernels with 64 rows per wave, head dims above 64 and up to 128 (fp16 and bf16).
#include "fa_bwd_wide.h"

// Compiled three times: as is for tensors whose head dim is 128, and with FA_PADDED = the columns to compute
// (128, or 96 for head dims up to that) for smaller head dims (a multiple of 8), where the kernels mask
// the excess columns.
#ifndef FA_PADDED
#define FA_PADDED 0
#endif
#if FA_PADDED == 96
#define FA_NAME(name) name##_cols96
#elif FA_PADDED
#define FA_NAME(name) name##_padded
#else
#define FA_NAME(name) name
#endif

namespace fa {
hipError_t FA_NAME(run_bwd_dkdv_wide_d128)(int dtype, const BwdArgs& a, bool windowed, hipStream_t s) {
  if (dtype == kDtypeBF16)
    return windowed ? launch_dkdv_wide<bf16_t, true, FA_PADDED>(a, s) : launch_dkdv_wide<bf16_t, false, FA_PADDED>(a, s);
  return windowed ? launch_dkdv_wide<f16_t, true, FA_PADDED>(a, s) : launch_dkdv_wide<f16_t, false, FA_PADDED>(a, s);
}
hipError_t FA_NAME(run_bwd_dq_wide_d128)(int dtype, const BwdArgs& a, bool windowed, hipStream_t s) {
  if (dtype == kDtypeBF16)
    return windowed ? launch_dq_wide<bf16_t, true, FA_PADDED>(a, s) : launch_dq_wide<bf16_t, false, FA_PADDED>(a, s);
  return windowed ? launch_dq_wide<f16_t, true, FA_PADDED>(a, s) : launch_dq_wide<f16_t, false, FA_PADDED>(a, s);
}
}  // namespace fa
