// Backward dq kernel instantiations for head dim 128 (fp16 and bf16).
#include "fa_bwd_impl.h"

// Compiled three times: as is for tensors whose head dim is 128, and with FA_PADDED = the columns to compute
// (128, or 96 for head dims up to that) for smaller head dims (a multiple of 8), where the kernels mask
// the excess columns.
#ifndef FA_PADDED
#define FA_PADDED 0
#endif
#if FA_PADDED == 96
#define FA_RUN run_bwd_dq_d128_cols96
#elif FA_PADDED
#define FA_RUN run_bwd_dq_d128_padded
#else
#define FA_RUN run_bwd_dq_d128
#endif

namespace fa {
hipError_t FA_RUN(int dtype, const BwdArgs& a, bool windowed, bool bias, bool dropout, hipStream_t s) {
  if (dtype == kDtypeBF16) return launch_bwd_dq<bf16_t, 128, FA_PADDED>(a, windowed, bias, dropout, s);
  return launch_bwd_dq<f16_t, 128, FA_PADDED>(a, windowed, bias, dropout, s);
}
}  // namespace fa
