// Instantiations of the forward for few query rows per K/V head, head dim 256 (fp16 and bf16).
#include "fa_fwd_rows.h"
#include "fa_kernels.h"

// Compiled twice, as the other per-head-dim files: FA_PADDED=256 for smaller head dims (a multiple of 8).
#ifndef FA_PADDED
#define FA_PADDED 0
#endif
#if FA_PADDED
#define FA_RUN run_fwd_rows_d256_padded
#else
#define FA_RUN run_fwd_rows_d256
#endif

namespace fa {
hipError_t FA_RUN(int dtype, const FwdArgs& a, bool windowed, bool bias, hipStream_t s) {
  if (dtype == kDtypeBF16) return launch_fwd_rows<bf16_t, 256, FA_PADDED != 0>(a, windowed, bias, s);
  return launch_fwd_rows<f16_t, 256, FA_PADDED != 0>(a, windowed, bias, s);
}
}  // namespace fa
