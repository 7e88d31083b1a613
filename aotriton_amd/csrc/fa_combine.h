// The second half of a forward whose keys are split over workgroups.
#pragma once
#include "fa_device.h"

namespace fa {

// Sums the parts of a row: out = sum_i 2^((m_i - m) sc) O_i / sum_i 2^((m_i - m) sc) l_i.
// Parts lie as (pair, row block, part, row of the block): a pair is `part_group` q-heads of one
// sequence, its rows are counted query * part_group + head and come in blocks of part_block.
// A thread takes four columns.  With many parts of few rows (packed rows: 896 at most) what bounds the sum is the
// latency of the loads, which miss L2 (other XCDs wrote them): a workgroup per row, whose threads hold all its parts between
// them and request sums and statistics together, so that one latency is left of several.  Few parts, or many rows, are bound by
// HBM: a thread has all parts of its columns, 256 / (D / 4) rows per workgroup, registers for eight waves a SIMD.
// One wave per row, statistics first, then eight parts at a time, took (us, old -> this): 17 parts of 32 rows D128 5.8 -> 4.6,
// 64 of 64 rows D64 6.5 -> 4.1; 2 parts of 32768 rows D128 21.2 -> 9.8 (42 MB), 8 of 18432 rows D64 10.0 -> 5.9.
struct CombineRow {
  int z, h, pq;            // sequence, q-head, query
  SeqInfo si;
  int64_t part;            // of the row in the first part
};
// row r of row block `block` (counted over all pairs); false where there is none
__device__ __forceinline__ bool combine_row(const FwdArgs& a, int block, int r, CombineRow& c) {
  const int group = a.part_group, per_seq = a.hq / group;
  const int rb = block % a.row_blocks, pair = block / a.row_blocks;
  if (r >= a.part_rows || pair * group >= a.num_zh) return false;
  const int hk = pair % per_seq, pr = rb * a.part_block + r;
  c.z = pair / per_seq;
  c.si = get_seq(a.seq, c.z);
  c.pq = pr / group;
  c.h = hk * group + pr % group;
  c.part = (int64_t)block * a.splits * a.part_rows + r;
  return c.pq < c.si.seqlen_q;
}
template <typename T>
__device__ __forceinline__ void combine_store(const FwdArgs& a, const CombineRow& c, int col, f32x4 acc, float m, float sc, float l) {
  const float inv = l > 0.f ? 1.0f / l : 0.f;
  if (col < a.head_dim_v) {
    vec<T, 4> t;
#pragma unroll
    for (int j = 0; j < 4; ++j) t[j] = Traits<T>::cvt(acc[j] * inv);
    *reinterpret_cast<vec<T, 4>*>(reinterpret_cast<T*>(a.out) + (int64_t)c.si.batch_index * a.so.z + (int64_t)c.h * a.so.h +
                                  (int64_t)(c.si.q_start + c.pq) * a.so.s + col) = t;
  }
  if (a.lse && col == 0) a.lse[lse_offset(c.si, c.h, a.hq) + c.pq] = lse_of(m, sc, l);
}

// A workgroup per row: more parts than kManyParts (its reduction through LDS costs what one more round of loads does) and no
// more rows than kManyRows, beyond which most of its threads have nothing to load and the rows come to thousands of workgroups (us,
// a workgroup per row / all parts in one thread: D64 11 parts of 768 rows 4.3 / 4.8, 10 of 6144 12.4 / 6.4, D128 10 of 96 4.2 / 4.5, of 768
// 5.1 / 5.1, of 4096 12.4 / 7.2).  Split tiles have at most kMostTileParts parts, packed rows with more never that many rows.
constexpr int kManyParts = 8, kMostTileParts = 16, kManyRows = 1024;

template <typename T, int D, int kParts>      // at most kParts parts, four of them in flight
static __global__ __launch_bounds__(256, 8) void combine_rows_kernel(const FwdArgs a) {
  constexpr int TPR = D / 4, ROWS = 256 / TPR;      // threads per row
  const int chunks = (a.part_rows + ROWS - 1) / ROWS;
  const int col = threadIdx.x % TPR * 4;
  CombineRow c;
  if (!combine_row(a, blockIdx.x / chunks, blockIdx.x % chunks * ROWS + threadIdx.x / TPR, c)) return;
  const float sc = score_scale(a.sm_scale, a.bias != nullptr);
  const float* po = a.part_o + c.part * D + col;
  const float* pm = a.part_ml + c.part * 2;
  vec<float, 2> ml[kParts];
#pragma unroll
  for (int i = 0; i < kParts; ++i)
    ml[i] = *reinterpret_cast<const vec<float, 2>*>(pm + (i < a.splits ? i : 0) * a.part_rows * 2);
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  float m, l = 0.f;
#pragma unroll
  for (int i0 = 0; i0 < kParts; i0 += 4) {
    constexpr int N = kParts < 4 ? kParts : 4;
    f32x4 x[N];
#pragma unroll
    for (int i = 0; i < N; ++i)
      x[i] = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(po + (i0 + i < a.splits ? i0 + i : 0) * a.part_rows * D));
    if (i0 == 0) {
      m = ml[0][0];
#pragma unroll
      for (int i = 1; i < kParts; ++i) m = fmaxf(m, ml[i][0]);
    }
#pragma unroll
    for (int i = 0; i < N; ++i) {
      // (a part in which the row saw no key has weight 0, and its sums may not have been written)
      const float f = i0 + i < a.splits && ml[i0 + i][1] != 0.f ? fast_exp2((ml[i0 + i][0] - m) * sc) : 0.f;
      l += f * ml[i0 + i][1];
      if (f != 0.f) acc += f * x[i];
    }
  }
  combine_store<T>(a, c, col, acc, m, sc, l);
}

// at most 64 parts
template <typename T, int D>
static __global__ __launch_bounds__(256, 4) void combine_many_kernel(const FwdArgs a) {
  constexpr int TPR = D / 4, SLOTS = 256 / TPR, PER = 64 / SLOTS;      // parts a thread may have
  __shared__ f32x4 s_acc[256];
  __shared__ float s_m[SLOTS], s_l[SLOTS];
  const int slot = threadIdx.x / TPR, col = threadIdx.x % TPR * 4;
  CombineRow c;
  if (!combine_row(a, blockIdx.x / a.part_rows, blockIdx.x % a.part_rows, c)) return;      // (the whole workgroup)
  const float sc = score_scale(a.sm_scale, a.bias != nullptr);
  const float* po = a.part_o + c.part * D + col;
  const float* pm = a.part_ml + c.part * 2;
  f32x4 x[PER];
  vec<float, 2> ml[PER];
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    // (past the last part: the first one's again, without weight)
    const int at = (slot + i * SLOTS < a.splits ? slot + i * SLOTS : 0) * a.part_rows;
    ml[i] = *reinterpret_cast<const vec<float, 2>*>(pm + at * 2);
    x[i] = *reinterpret_cast<const f32x4*>(po + at * D);
  }
  float m = ml[0][0];
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    m = fmaxf(m, ml[i][0]);
    if (slot + i * SLOTS >= a.splits) ml[i][1] = 0.f;
  }
  if (col == 0) s_m[slot] = m;
  __syncthreads();
#pragma unroll
  for (int i = 0; i < SLOTS; ++i) m = fmaxf(m, s_m[i]);
  float l = 0.f;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const float f = ml[i][1] != 0.f ? fast_exp2((ml[i][0] - m) * sc) : 0.f;
    l += f * ml[i][1];
    if (f != 0.f) acc += f * x[i];
  }
  s_acc[threadIdx.x] = acc;
  if (col == 0) s_l[slot] = l;
  __syncthreads();
  if (slot != 0) return;
  l = s_l[0];
#pragma unroll
  for (int i = 1; i < SLOTS; ++i) {
    l += s_l[i];
    acc += s_acc[i * TPR + threadIdx.x];
  }
  combine_store<T>(a, c, col, acc, m, sc, l);
}

template <typename T, int D>
hipError_t launch_combine_rows(const FwdArgs& a, int pairs, hipStream_t stream) {
  const int64_t blocks = (int64_t)pairs * a.row_blocks;
  if (blocks * a.part_rows == 0) return hipSuccess;
  constexpr int ROWS = 256 / (D / 4);
  if (a.splits > kMostTileParts || (a.splits > kManyParts && blocks * a.part_rows <= kManyRows))
    hipLaunchKernelGGL((combine_many_kernel<T, D>), dim3((unsigned)(blocks * a.part_rows)), dim3(256), 0, stream, a);
  else
    hipLaunchKernelGGL((a.splits > kManyParts ? combine_rows_kernel<T, D, kMostTileParts>
                        : a.splits > 2 ? combine_rows_kernel<T, D, kManyParts> : combine_rows_kernel<T, D, 2>),
                       dim3((unsigned)(blocks * ((a.part_rows + ROWS - 1) / ROWS))), dim3(256), 0, stream, a);
  return hipGetLastError();
}

}  // namespace fa
