// The second half of a forward whose keys are split over workgroups.
#pragma once
#include "fa_device.h"

namespace fa {

// Sums the parts of a row: out = sum_i 2^((m_i - m) sc) O_i / sum_i 2^((m_i - m) sc) l_i, one wave per row.
// Parts lie as (pair, row block, part, row of the block): a pair is `part_group` q-heads of one
// sequence, its rows are counted query * part_group + head and come in blocks of part_block.  What
// bounds it is the latency of its loads: the statistics of all parts in one load, the sums eight parts
// at a time (one part after the other it took 6.5 us for 17 parts of 32 rows, as long as the kernel
// before it).
template <typename T, int D>
static __global__ __launch_bounds__(256) void combine_rows_kernel(const FwdArgs a) {
  constexpr int PL = D / 64;      // columns per lane
  const int group = a.part_group;
  const int lane = threadIdx.x & 63;
  const int item = blockIdx.x * 4 + (threadIdx.x >> 6);      // (pair, row block, row)
  const int r = item % a.part_rows, block = item / a.part_rows;
  const int rb = block % a.row_blocks, pair = block / a.row_blocks;
  if (pair * group >= a.num_zh) return;
  const int per_seq = a.hq / group;
  const int z = pair / per_seq, hk = pair % per_seq;
  const SeqInfo si = get_seq(a.seq, z);
  const int pr = rb * a.part_block + r;
  if (pr >= si.seqlen_q * group) return;
  const int64_t part = (int64_t)block * a.splits * a.part_rows + r;
  // lane i holds split i's maximum and row sum (at most 64 splits)
  float ms = -__builtin_inff(), ls = 0.f;
  if (lane < a.splits) {
    const vec<float, 2> t = *reinterpret_cast<const vec<float, 2>*>(a.part_ml + (part + (int64_t)lane * a.part_rows) * 2);
    ms = t[0]; ls = t[1];
  }
  const float sc = score_scale(a.sm_scale, a.bias != nullptr);
  float m = ms;
#pragma unroll
  for (int d = 32; d >= 1; d /= 2) m = fmaxf(m, __shfl_xor(m, d));
  const float f = ls != 0.f ? fast_exp2((ms - m) * sc) : 0.f;
  float lsum = f * ls;
#pragma unroll
  for (int d = 32; d >= 1; d /= 2) lsum += __shfl_xor(lsum, d);
  const float* po = a.part_o + part * D + lane * PL;
  const int64_t step = (int64_t)a.part_rows * D;
  vec<float, PL> acc;
#pragma unroll
  for (int j = 0; j < PL; ++j) acc[j] = 0.f;
  for (int i0 = 0; i0 < a.splits; i0 += 8) {      // eight loads in flight
    vec<float, PL> x[8];
#pragma unroll
    for (int u = 0; u < 8; ++u)
      x[u] = *reinterpret_cast<const vec<float, PL>*>(po + (i0 + u < a.splits ? i0 + u : i0) * step);
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (i0 + u < a.splits) {
        // (a part in which the row saw no key has weight 0, and its sums may not have been written)
        const float fu = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, f), i0 + u));
        if (fu != 0.f) acc += fu * x[u];
      }
  }
  const int pq = pr / group, ph = hk * group + pr % group;
  const bool alive = lsum > 0.f;
  const float inv = alive ? 1.0f / lsum : 0.f;
  T* op = reinterpret_cast<T*>(a.out) + (int64_t)si.batch_index * a.so.z + (int64_t)ph * a.so.h +
          (int64_t)(si.q_start + pq) * a.so.s + lane * PL;
  if (lane * PL < a.head_dim_v) {
    vec<T, PL> t;
#pragma unroll
    for (int j = 0; j < PL; ++j) t[j] = Traits<T>::cvt(acc[j] * inv);
    *reinterpret_cast<vec<T, PL>*>(op) = t;
  }
  if (a.lse && lane == 0) a.lse[lse_offset(si, ph, a.hq) + pq] = lse_of(m, sc, lsum);
}

template <typename T, int D>
hipError_t launch_combine_rows(const FwdArgs& a, int pairs, hipStream_t stream) {
  const int64_t rows = (int64_t)pairs * a.row_blocks * a.part_rows;
  if (rows == 0) return hipSuccess;
  hipLaunchKernelGGL((combine_rows_kernel<T, D>), dim3((unsigned)((rows + 3) / 4)), dim3(256), 0, stream, a);
  return hipGetLastError();
}

}  // namespace fa
