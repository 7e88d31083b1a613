// Forward kernels with dropout for head dim 256 (fp16 and bf16).  A file of its own for its compiler option (build.py): with the
// scores in vector registers these kernels take 1-3 % less time, and the one with a bias and a window but no dropout 3 % more.
#include "fa_fwd_impl.h"

// Compiled twice, as fa_fwd_d256.hip is.
#ifndef FA_PADDED
#define FA_PADDED 0
#endif

namespace fa {
#define FA_DROPOUT(T)                                                                                        \
  template hipError_t launch_fwd_variant<T, 256, false, false, true, FA_PADDED>(const FwdArgs&, dim3, hipStream_t); \
  template hipError_t launch_fwd_variant<T, 256, false, true, true, FA_PADDED>(const FwdArgs&, dim3, hipStream_t);  \
  template hipError_t launch_fwd_variant<T, 256, true, false, true, FA_PADDED>(const FwdArgs&, dim3, hipStream_t);  \
  template hipError_t launch_fwd_variant<T, 256, true, true, true, FA_PADDED>(const FwdArgs&, dim3, hipStream_t);
FA_DROPOUT(f16_t)
FA_DROPOUT(bf16_t)
}  // namespace fa
