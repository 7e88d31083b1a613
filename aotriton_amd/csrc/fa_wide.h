// What the kernels with 64 rows per wave share (fa_bwd_wide.h, fa_fwd_wide.h).
#pragma once
#include <type_traits>

#include "fa_device.h"

namespace fa {

// One MFMA onto an accumulator that stays in accumulation registers.  What the compiler sees to for its own MFMAs (its hazard
// recognizer does not look into an asm statement) is arranged by the callers: the conversions that make a B operand are at
// least two instructions back (s_nop where a phase begins; `build --scan` checks the compiler's output for it), and the
// accumulators are touched by nothing else inside the loops and read behind acc_settle only.
template <typename T> __device__ __forceinline__ void mfma_acc(f32x16& c, typename Traits<T>::op_t a, typename Traits<T>::op_t b);
template <> __device__ __forceinline__ void mfma_acc<bf16_t>(f32x16& c, Traits<bf16_t>::op_t a, Traits<bf16_t>::op_t b) {
  asm("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
}
template <> __device__ __forceinline__ void mfma_acc<f16_t>(f32x16& c, Traits<f16_t>::op_t a, Traits<f16_t>::op_t b) {
  asm("v_mfma_f32_32x32x16_f16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
}

// An accumulator of zeros, made by the matrix pipe as well (through vector registers it would take as many of those).
template <typename T> __device__ __forceinline__ void acc_zero(f32x16& c) {
  const u32x4_t z = {0, 0, 0, 0};
  if constexpr (std::is_same<T, bf16_t>::value) asm volatile("s_nop 1\n\tv_mfma_f32_32x32x16_bf16 %0, %1, %1, 0" : "=a"(c) : "v"(z));
  else asm volatile("s_nop 1\n\tv_mfma_f32_32x32x16_f16 %0, %1, %1, 0" : "=a"(c) : "v"(z));
}
// Waits until the MFMAs have written the accumulators (16 passes and what the register file takes).
template <int N> __device__ __forceinline__ void acc_settle(f32x16 (&x)[N], f32x16 (&y)[N]) {
  if constexpr (N == 4)
    asm volatile("s_nop 15\n\ts_nop 15" : "+a"(x[0]), "+a"(x[1]), "+a"(x[2]), "+a"(x[3]), "+a"(y[0]), "+a"(y[1]), "+a"(y[2]), "+a"(y[3]));
  else
    asm volatile("s_nop 15\n\ts_nop 15" : "+a"(x[0]), "+a"(x[1]), "+a"(x[2]), "+a"(y[0]), "+a"(y[1]), "+a"(y[2]));
}

// A wave's 1 KB of a tile straight into LDS (64 lanes x 16 bytes at voff + soff, to lds + 16 lane).  The compiler's builtin
// does the same but makes the first transposing LDS read behind it wait for it; here the tile's one wait is placed by hand.
__device__ __forceinline__ void load_to_lds(u32x4_t rsrc, int voff, int soff, int lds) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
               :: "s"(lds), "v"(voff), "s"(rsrc), "s"(soff) : "m0");
}
// (lengths that were loaded arrive in vector registers, and the arithmetic on them stays there unless told otherwise)
__device__ __forceinline__ SeqInfo uniform(SeqInfo s) {
  s.seqlen_q = __builtin_amdgcn_readfirstlane(s.seqlen_q); s.seqlen_k = __builtin_amdgcn_readfirstlane(s.seqlen_k);
  s.q_start = __builtin_amdgcn_readfirstlane(s.q_start); s.k_start = __builtin_amdgcn_readfirstlane(s.k_start);
  return s;
}
template <typename V> __device__ __forceinline__ V lds_read(int at) {
  return *reinterpret_cast<__attribute__((address_space(3))) const V*>(at);
}
__device__ __forceinline__ tr_raw_t lds_read_tr_at(int at) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16(reinterpret_cast<__attribute__((address_space(3))) tr_raw_t*>(at));
}
__device__ __forceinline__ int lds_offset(const void* p) { return (int)(uintptr_t)(__attribute__((address_space(3))) const void*)p; }

}  // namespace fa
