// Host-visible launchers of the gfx950 kernels (one translation unit per head dim).
#pragma once
#include <hip/hip_runtime.h>

#include "fa_args.h"

namespace fa {

constexpr int kDtypeF32 = 1, kDtypeF16 = 2, kDtypeBF16 = 3;

struct TileShape { int block_m, block_n, num_waves, lds_bytes, per_cu = 1; };   // per_cu: persistent workgroups per CU

hipError_t run_fwd_d64(int dtype, const FwdArgs& a, bool windowed, bool bias, bool dropout, hipStream_t s);
hipError_t run_fwd_d128(int dtype, const FwdArgs& a, bool windowed, bool bias, bool dropout, hipStream_t s);
hipError_t run_fwd_d256(int dtype, const FwdArgs& a, bool windowed, bool bias, bool dropout, hipStream_t s);
// the same kernels with the columns past FwdArgs::head_dim masked (head dims rounded up)
hipError_t run_fwd_d64_padded(int dtype, const FwdArgs& a, bool windowed, bool bias, bool dropout, hipStream_t s);
hipError_t run_fwd_d128_padded(int dtype, const FwdArgs& a, bool windowed, bool bias, bool dropout, hipStream_t s);
// Head dims above 64 and up to 96 (both of them) compute 96 columns in the 128-column layout: a quarter of the
// matrix work and of the operand reads were zeros (bf16, B4 H32 S4096 D96: forward 522 -> 459 us causal, 928 -> 813
// full, backward 1726 -> 1572 causal; with dropout, bound by the vector ALU, 2 %).  Same sums: what is left out is zero.
hipError_t run_fwd_d128_cols96(int dtype, const FwdArgs& a, bool windowed, bool bias, bool dropout, hipStream_t s);
hipError_t run_fwd_d256_padded(int dtype, const FwdArgs& a, bool windowed, bool bias, bool dropout, hipStream_t s);
// head dims above 64 and up to 128 without bias and dropout, a positive scale: 64 rows per wave (fa_fwd_wide.h)
hipError_t run_fwd_wide_d128(int dtype, const FwdArgs& a, bool windowed, hipStream_t s);
hipError_t run_fwd_wide_d128_padded(int dtype, const FwdArgs& a, bool windowed, hipStream_t s);
hipError_t run_fwd_wide_d128_cols96(int dtype, const FwdArgs& a, bool windowed, hipStream_t s);
inline hipError_t run_fwd_wide(int dtype, const FwdArgs& a, bool windowed, hipStream_t s) {
  if (a.head_dim == 128 && a.head_dim_v == 128) return run_fwd_wide_d128(dtype, a, windowed, s);
  return (a.head_dim <= 96 && a.head_dim_v <= 96 ? run_fwd_wide_d128_cols96 : run_fwd_wide_d128_padded)(dtype, a, windowed, s);
}
TileShape fwd_wide_shape();
// few query rows per K/V head: packed rows of a GQA group, keys split over workgroups (fa_fwd_rows.h)
hipError_t run_fwd_rows_d64(int dtype, const FwdArgs& a, bool windowed, bool bias, hipStream_t s);
hipError_t run_fwd_rows_d128(int dtype, const FwdArgs& a, bool windowed, bool bias, hipStream_t s);
hipError_t run_fwd_rows_d256(int dtype, const FwdArgs& a, bool windowed, bool bias, hipStream_t s);
hipError_t run_fwd_rows_d64_padded(int dtype, const FwdArgs& a, bool windowed, bool bias, hipStream_t s);
hipError_t run_fwd_rows_d128_padded(int dtype, const FwdArgs& a, bool windowed, bool bias, hipStream_t s);
hipError_t run_fwd_rows_d256_padded(int dtype, const FwdArgs& a, bool windowed, bool bias, hipStream_t s);
// tile table lookups: (element type, head dim, causal / windowed) and the variant
TileShape fwd_tile_shape(int dtype, int head_dim, bool windowed, int half_tiles);

hipError_t run_encoded_softmax(const EncodedSoftmaxArgs& a, hipStream_t s);
// strided -> packed (unpack false) or packed -> strided (unpack true); elem_bytes 2 or 4
hipError_t run_repack(int elem_bytes, bool unpack, const RepackArgs& a, hipStream_t s);
// `count` words of host memory to device memory, as kernel arguments
hipError_t run_write_words(uint32_t* dst, const uint32_t* words, int count, hipStream_t s);
// register-only MFMA loop: the rate the matrix pipe sustains (benchmark aid)
hipError_t run_mfma_rate(bool random_operands, int grid, int iters, float* out, unsigned long long* clk, hipStream_t s);

// backward: kernel_slot 0 = preprocess (delta), 1 = dK/dV, 2 = dQ, 3 = fused
hipError_t run_bwd_preprocess(int dtype, int head_dim, const BwdArgs& a, hipStream_t s);
hipError_t run_bwd_dkdv(int dtype, int head_dim, const BwdArgs& a, bool windowed, bool bias, bool dropout, hipStream_t s);
// the same with the items cut into parts and a kernel behind it that adds the parts up (BwdArgs::part_ws)
hipError_t run_bwd_dkdv_parts(int dtype, int head_dim, const BwdArgs& a, bool windowed, bool bias, bool dropout, hipStream_t s);
// Every row of the bias is whole 16-byte pieces at 16-byte boundaries, in every item.
inline bool plain_bias(const BwdArgs& a) {
  return a.seq.num_seqlens == 0 && a.seq.max_seqlen_k % 8 == 0 && bias_aligned(a.bias, a.sb_z, a.sb_h, a.sb_m, a.sb_n);
}
// The same for items that store dS at head dims above 128, whole or in parts, without a bias or with a plain one: pairs of waves
// (fa_bwd_pair.h).
inline bool bwd_dkdv_by_pairs(const BwdArgs& a, int head_dim, bool bias, bool stored_ds) {
  return stored_ds && head_dim == 256 && (!bias || plain_bias(a));
}
hipError_t run_bwd_dkdv_pair(int dtype, const BwdArgs& a, bool windowed, bool bias, bool dropout, hipStream_t s);
TileShape bwd_pair_shape(bool bias);
hipError_t run_bwd_dq(int dtype, int head_dim, const BwdArgs& a, bool windowed, bool bias, bool dropout, hipStream_t s);
// head dims above 64 and up to 128 without bias and dropout: 64 rows per wave (fa_bwd_wide.h)
hipError_t run_bwd_dkdv_wide(int dtype, const BwdArgs& a, bool windowed, hipStream_t s);
hipError_t run_bwd_dq_wide(int dtype, const BwdArgs& a, bool windowed, hipStream_t s);
TileShape bwd_wide_shape(bool dkdv);
hipError_t run_bwd_fused(int dtype, int head_dim, const BwdArgs& a, bool windowed, bool bias, bool dropout, hipStream_t s);
TileShape bwd_tile_shape(int dtype, int head_dim, bool windowed, bool bias, bool dropout, int kernel_slot, bool stored_ds);
// dQ = dS K from the dS tiles that the dK/dV kernel stored (BwdArgs::ds_ws), and their geometry
hipError_t run_bwd_dqs(int dtype, int head_dim, const BwdArgs& a, hipStream_t s);
void ds_tile_counts(int head_dim, int max_sq, int max_sk, int* ntq, int* ntk, int64_t* tile_bytes);

// MFMA kernels of the 16-bit types for head dims above 256, rounded up to 512 (the head dim split
// over the waves of a workgroup).  kernel_slot of the backward: 1 dK/dV, 2 dQ and dB.
hipError_t run_fwd_d512(int dtype, const FwdArgs& a, bool windowed, bool bias, bool dropout, hipStream_t s);
hipError_t run_bwd_d512(int dtype, int kernel_slot, const BwdArgs& a, bool windowed, bool bias, bool dropout,
                        hipStream_t s);
TileShape d512_tile_shape(int kernel_slot);

// MFMA kernels for fp32 tensors at head dims up to 256 (compiled for 128 and 256 columns, the head
// dim split over the waves of a workgroup).  kernel_slot of the backward: 1 dK/dV, 2 dQ and dB.
hipError_t run_fwd_f32(int head_dim, const FwdArgs& a, bool windowed, bool bias, bool dropout, hipStream_t s);
hipError_t run_bwd_f32(int head_dim, int kernel_slot, const BwdArgs& a, bool windowed, bool bias, bool dropout,
                       hipStream_t s);
// fp32, head dims up to 128 (compiled for 64 and 128 columns): four waves share 32 rows and split the other
// side.  kernel_slot 2 also writes delta; kernel_slot 1 reads it.
hipError_t run_fwd_f32_rows(int head_dim, const FwdArgs& a, bool windowed, bool bias, bool dropout, hipStream_t s);
hipError_t run_bwd_f32_rows(int head_dim, int kernel_slot, const BwdArgs& a, bool windowed, bool bias, bool dropout,
                            hipStream_t s);
TileShape f32_rows_tile_shape(int head_dim);
TileShape f32_tile_shape(int head_dim, int kernel_slot);

// Vector-ALU kernels (no MFMA): every type at every compiled head dim; they serve tensors whose
// rows the MFMA kernels cannot load in 16-byte pieces, and delta of the fp32 and split-head-dim families.
// head_dim is the compiled one (64, 128, 256, 512).  kernel_slot of the backward: 0 delta,
// 1 dK/dV, 2 dQ and dB.
hipError_t run_fwd_valu(int dtype, int head_dim, const FwdArgs& a, hipStream_t s);
hipError_t run_bwd_valu(int dtype, int head_dim, int kernel_slot, const BwdArgs& a, hipStream_t s);

}  // namespace fa
