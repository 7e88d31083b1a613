// Forward with 64 rows per wave, head dims above 64 and up to 128 (fp16 and bf16).
#include "fa_fwd_wide.h"
#include "fa_kernels.h"

// Compiled three times: as is for tensors whose head dim is 128, and with FA_PADDED = the columns to compute
// (128, or 96 for head dims up to that) for smaller head dims (a multiple of 8), where the kernels mask
// the excess columns.
#ifndef FA_PADDED
#define FA_PADDED 0
#endif
#if FA_PADDED == 96
#define FA_RUN run_fwd_wide_d128_cols96
#elif FA_PADDED
#define FA_RUN run_fwd_wide_d128_padded
#else
#define FA_RUN run_fwd_wide_d128
#endif

namespace fa {
hipError_t FA_RUN(int dtype, const FwdArgs& a, bool windowed, hipStream_t s) {
  return dtype == kDtypeBF16 ? launch_fwd_wide_any<bf16_t, FA_PADDED>(a, windowed, s) : launch_fwd_wide_any<f16_t, FA_PADDED>(a, windowed, s);
}
}  // namespace fa
