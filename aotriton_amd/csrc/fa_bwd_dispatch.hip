// Head-dim dispatch of the backward launchers and the delta (preprocess) kernel.
#include "fa_bwd_impl.h"

namespace fa {

// Tensors whose head dim is one of the compiled ones take the kernels with a constant head
// dim; smaller head dims take the copies that mask the excess columns, of 96 computed columns where both head
// dims fit (see run_fwd_d128_cols96; `upto96` names that copy, the padded one where there is none).
#define FA_DECL(name, upto96)                                                                           \
  hipError_t name##_d64(int, const BwdArgs&, bool, bool, bool, hipStream_t);                            \
  hipError_t name##_d128(int, const BwdArgs&, bool, bool, bool, hipStream_t);                           \
  hipError_t name##_d256(int, const BwdArgs&, bool, bool, bool, hipStream_t);                           \
  hipError_t name##_d64_padded(int, const BwdArgs&, bool, bool, bool, hipStream_t);                     \
  hipError_t name##_d128_padded(int, const BwdArgs&, bool, bool, bool, hipStream_t);                    \
  hipError_t name##_d128_##upto96(int, const BwdArgs&, bool, bool, bool, hipStream_t);                  \
  hipError_t name##_d256_padded(int, const BwdArgs&, bool, bool, bool, hipStream_t);                    \
  hipError_t name(int dtype, int head_dim, const BwdArgs& a, bool w, bool b, bool p, hipStream_t s) {   \
    const bool padded = a.head_dim != head_dim || a.head_dim_v != head_dim;                             \
    switch (head_dim) {                                                                                 \
      case 64: return padded ? name##_d64_padded(dtype, a, w, b, p, s) : name##_d64(dtype, a, w, b, p, s);    \
      case 128:                                                                                         \
        if (a.head_dim <= 96 && a.head_dim_v <= 96) return name##_d128_##upto96(dtype, a, w, b, p, s);  \
        return padded ? name##_d128_padded(dtype, a, w, b, p, s) : name##_d128(dtype, a, w, b, p, s);   \
      case 256: return padded ? name##_d256_padded(dtype, a, w, b, p, s) : name##_d256(dtype, a, w, b, p, s); \
    }                                                                                                   \
    return hipErrorNotSupported;                                                                        \
  }

FA_DECL(run_bwd_dkdv, cols96)
FA_DECL(run_bwd_dkdv_parts, padded)
FA_DECL(run_bwd_dq, cols96)
FA_DECL(run_bwd_fused, padded)
#undef FA_DECL

hipError_t run_bwd_dkdv_pair_d256(int, const BwdArgs&, bool, bool, bool, hipStream_t);
hipError_t run_bwd_dkdv_pair_d256_padded(int, const BwdArgs&, bool, bool, bool, hipStream_t);
hipError_t run_bwd_dkdv_pair(int dtype, const BwdArgs& a, bool w, bool b, bool p, hipStream_t s) {
  const bool padded = a.head_dim != 256 || a.head_dim_v != 256;
  return (padded ? run_bwd_dkdv_pair_d256_padded : run_bwd_dkdv_pair_d256)(dtype, a, w, b, p, s);
}

#define FA_DECL_WIDE(name)                                                                    \
  hipError_t name##_d128(int, const BwdArgs&, bool, hipStream_t);                             \
  hipError_t name##_d128_padded(int, const BwdArgs&, bool, hipStream_t);                      \
  hipError_t name##_d128_cols96(int, const BwdArgs&, bool, hipStream_t);                      \
  hipError_t name(int dtype, const BwdArgs& a, bool w, hipStream_t s) {                       \
    if (a.head_dim == 128 && a.head_dim_v == 128) return name##_d128(dtype, a, w, s);         \
    const bool upto96 = a.head_dim <= 96 && a.head_dim_v <= 96;                               \
    return upto96 ? name##_d128_cols96(dtype, a, w, s) : name##_d128_padded(dtype, a, w, s);  \
  }
FA_DECL_WIDE(run_bwd_dkdv_wide)
FA_DECL_WIDE(run_bwd_dq_wide)
#undef FA_DECL_WIDE

hipError_t run_bwd_preprocess(int dtype, int head_dim, const BwdArgs& a, hipStream_t s) {
  const bool bf = dtype == kDtypeBF16;
  switch (head_dim) {
    case 64: return bf ? launch_bwd_preprocess<bf16_t, 64>(a, s) : launch_bwd_preprocess<f16_t, 64>(a, s);
    case 128: return bf ? launch_bwd_preprocess<bf16_t, 128>(a, s) : launch_bwd_preprocess<f16_t, 128>(a, s);
    case 256: return bf ? launch_bwd_preprocess<bf16_t, 256>(a, s) : launch_bwd_preprocess<f16_t, 256>(a, s);
  }
  return hipErrorNotSupported;
}

}  // namespace fa
