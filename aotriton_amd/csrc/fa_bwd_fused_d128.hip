// Backward fused kernel instantiations for head dim 128 (fp16 and bf16).
#include "fa_bwd_fused_impl.h"

// Compiled twice: as is for tensors whose head dim is 128, and with FA_PADDED = the columns to compute for smaller
// head dims (a multiple of 8), where the kernels mask the excess columns.
#ifndef FA_PADDED
#define FA_PADDED 0
#endif
#if FA_PADDED
#define FA_RUN run_bwd_fused_d128_padded
#else
#define FA_RUN run_bwd_fused_d128
#endif

namespace fa {
hipError_t FA_RUN(int dtype, const BwdArgs& a, bool windowed, bool bias, bool dropout, hipStream_t s) {
  if (dtype == kDtypeBF16) return launch_bwd_fused<bf16_t, 128, FA_PADDED>(a, windowed, bias, dropout, s);
  return launch_bwd_fused<f16_t, 128, FA_PADDED>(a, windowed, bias, dropout, s);
}
}  // namespace fa
