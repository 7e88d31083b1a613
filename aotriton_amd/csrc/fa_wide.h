// What the kernels with 64 rows per wave (fa_bwd_wide.h, fa_fwd_wide.h) and those of pairs of waves (fa_bwd_pair.h, fa_fwd_pair.h) share.
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

// The rescaling of an O^T accumulator tuple (a lane's 16 values times its row's factor) in place in
// the accumulation registers: the tuple never shows up in VGPRs.  The waits cover the hazards that
// nobody checks inside an asm block: an MFMA result read by the vector ALU (up to 19 wait states)
// and a vector write read by an MFMA as its C operand.
#define FA_ACC_OPS(m) m(0) m(1) m(2) m(3) m(4) m(5) m(6) m(7) m(8) m(9) m(10) m(11) m(12) m(13) m(14) m(15)
#define FA_ACC_SCALE1(i) "v_accvgpr_read_b32 %16, %" #i "\n v_mul_f32 %16, %16, %17\n v_accvgpr_write_b32 %" #i ", %16\n"
#define FA_ACC_SPLIT(t) \
  float e0 = t[0], e1 = t[1], e2 = t[2], e3 = t[3], e4 = t[4], e5 = t[5], e6 = t[6], e7 = t[7], e8 = t[8], e9 = t[9], \
        e10 = t[10], e11 = t[11], e12 = t[12], e13 = t[13], e14 = t[14], e15 = t[15]
#define FA_ACC_JOIN(t) \
  t[0] = e0; t[1] = e1; t[2] = e2; t[3] = e3; t[4] = e4; t[5] = e5; t[6] = e6; t[7] = e7; t[8] = e8; t[9] = e9; \
  t[10] = e10; t[11] = e11; t[12] = e12; t[13] = e13; t[14] = e14; t[15] = e15
__device__ __forceinline__ void acc_scale(f32x16& t, float f) {
  float tmp;
  FA_ACC_SPLIT(t);
  asm volatile("s_nop 15\n s_nop 7\n" FA_ACC_OPS(FA_ACC_SCALE1) "s_nop 3\n"
               : "+a"(e0), "+a"(e1), "+a"(e2), "+a"(e3), "+a"(e4), "+a"(e5), "+a"(e6), "+a"(e7), "+a"(e8), "+a"(e9),
                 "+a"(e10), "+a"(e11), "+a"(e12), "+a"(e13), "+a"(e14), "+a"(e15), "=&v"(tmp)
               : "v"(f));
  FA_ACC_JOIN(t);
}

// Twice a wave's 1 KB of a tile straight into LDS (64 lanes x 16 bytes at voff + soff, to lds + 16 lane).  The compiler's builtin
// does the same but makes the first transposing LDS read behind it wait for it; here the tile's one wait is placed by hand.
// A scalar register that a vector instruction has written (v_readfirstlane, the v_readlane that brings a spilled one back) may be
// read by a memory instruction five wait states later.  The compiler sees to it for its own and does not look into asm: the
// move and s_nop 3 are the five, whatever stands in front; two loads share them.
__device__ __forceinline__ void load_to_lds(u32x4_t rsrc, int voff0, int soff0, int lds0, int voff1, int soff1, int lds1) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 3\n\tbuffer_load_dwordx4 %2, %4, %5 offen lds\n\t"
               "s_mov_b32 m0, %1\n\ts_nop 0\n\tbuffer_load_dwordx4 %3, %4, %6 offen lds"
               :: "s"(lds0), "s"(lds1), "v"(voff0), "v"(voff1), "s"(rsrc), "s"(soff0), "s"(soff1) : "m0");
}
// A wave's 64 x 16 bytes straight into LDS (see load_to_lds).
__device__ __forceinline__ void load_to_lds1(u32x4_t rsrc, int voff, int lds) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 3\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds" :: "s"(lds), "v"(voff), "s"(rsrc) : "m0");
}
// Two consecutive KB that nobody reads again.
__device__ __forceinline__ void load_to_lds_once(u32x4_t rsrc, int voff0, int voff1, int soff, int lds) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 3\n\tbuffer_load_dwordx4 %2, %4, %5 offen nt lds\n\t"
               "s_mov_b32 m0, %1\n\ts_nop 0\n\tbuffer_load_dwordx4 %3, %4, %6 offen nt lds"
               :: "s"(lds), "s"(lds + 1024), "v"(voff0), "v"(voff1), "s"(rsrc), "s"(soff), "s"(soff + 1024) : "m0");
}
// Accesses i and i + 1 of the 16 that bring a wave's 64 rows of 128 columns into LDS (swizzled; a lane's row of access 0 is `voff`
// bytes from the first, the rows of two accesses `step` apart; chunks past column d are zero).
__device__ __forceinline__ void rows_to_lds(u32x4_t rsrc, int voff, int step, int d, int lds, int i) {
  const int lane = threadIdx.x & 63, row4 = lane / 16, ch = lane % 16;
  const int c0 = ch ^ Swz<128>::f(row4 + 4 * i), c1 = ch ^ Swz<128>::f(row4 + 4 * i + 4);
  load_to_lds(rsrc, c0 * 8 < d ? voff + c0 * 16 : kVoffOutOfRange, i * step, lds + i * 1024,
              c1 * 8 < d ? voff + c1 * 16 : kVoffOutOfRange, (i + 1) * step, lds + (i + 1) * 1024);
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
template <typename V> __device__ __forceinline__ void lds_write(int at, V x) {
  *reinterpret_cast<__attribute__((address_space(3))) V*>(at) = x;
}
__device__ __forceinline__ tr_raw_t lds_read_tr_at(int at) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16(reinterpret_cast<__attribute__((address_space(3))) tr_raw_t*>(at));
}
__device__ __forceinline__ int lds_offset(const void* p) { return (int)(uintptr_t)(__attribute__((address_space(3))) const void*)p; }

}  // namespace fa
