// MFMA kernels for fp32 tensors of head dims up to 128 (v_mfma_f32_32x32x2_f32), gfx950.
//
// They compute what fa_f32.hip describes, in fp32 throughout, with another split of the work: the
// four waves of a workgroup own the SAME 32 rows (queries; keys in the dK/dV kernel) with the whole head
// dim, and each takes every fourth 32-row block of the other side.  Nothing is shared until the end,
// when the waves' sums meet in LDS: no barrier, no tile staging and no partial blocks in the loop.
//
// What bounds them: the fp32 matrix pipe.  A block costs a wave D MFMAs (forward; 1.5 D in dQ, 2 D in
// dK/dV) of 64 cycles, against 8 D bytes of operands per row of the block, so every operand comes
// straight from L1 / L2 in the layout the MFMA wants: as the row operand a lane's 16-byte pieces of
// row lane % 32 (columns 8 j + 4 hi + 0..3, four MFMAs each), as the transposed operand single floats, a wave
// reading 32 consecutive ones of two rows.  The registers that held one block's row operand take
// the next operand as soon as its MFMAs are issued, so a load has one GEMM (1-2 us) to arrive.
// Two waves per SIMD at 64 columns, one at 128.  Measured (one box, against fa_f32.hip): D = 64, where
// those kernels multiply 64 columns of zeros: B4 H32 S4096 forward 9.48 -> 4.45 ms (123 TFLOP/s of the 157
// that the fp32 MFMA gives), backward 33.3 -> 14.6; B2 H4 S128 14.9 -> 7.2 us and 36 -> 19.  D = 128: forward
// level on large batches, 56 -> 31 us at H12 S600; backward slower once the chip is full (dK/dV 1.62 against
// 1.25 ms at B2 H16 S2048), 10 % faster on small ones: fa_api.cpp has the rule.
// Splitting the other side over the waves also gives short sequences and small batches four waves per
// 32 rows where fa_f32.hip has one per 8 rows of a tile in lockstep.
#include "fa_device.h"
#include "fa_kernels.h"

namespace fa {
namespace {

constexpr int kWaves = 4;

// Between the phases of a block: a load issued behind one of these stays behind it (the compiler would
// otherwise request every operand of a block up front and spill them).
__device__ __forceinline__ void phase() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

template <int D>
struct FR {
  static constexpr int KJ = D / 8;          // 16-byte pieces of a row per lane
  static constexpr int DB = D / 32;         // 32-column blocks
  static constexpr int OSTR = D + 4;        // floats per row of a wave's sums in LDS
  static constexpr int AREA = 32 * OSTR;    // floats per wave
  static constexpr int SMEM = kWaves * (AREA + 64) * 4;
};

__device__ __forceinline__ f32x16 mfma_f32(float a, float b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}

// A block of 32 rows of one tensor: descriptor bounded to its valid rows, per-lane offsets of both operand forms.
template <int D>
struct Block {
  const float* base;      // row 0 of the sequence
  int64_t stride;
  int rows, cols;         // rows of the sequence, columns of the tensor
  int c, hi;
  __device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc(int b) const {
    const int n = rows - b * 32 < 32 ? rows - b * 32 : 32;
    return wave_rsrc(base + (int64_t)b * 32 * stride, n > 0 ? ((n - 1) * (int)stride + cols) * 4 : 0);
  }
  // row operand: columns past the tensor's read as zero
  __device__ __forceinline__ void load_rows(f32x4 (&x)[FR<D>::KJ], int b) const {
    const auto rs = rsrc(b);
    const int at = c * (int)stride * 4 + hi * 16;
#pragma unroll
    for (int j = 0; j < FR<D>::KJ; ++j)
      x[j] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                           rs, 8 * j + 4 * hi < cols ? at + 32 * j : kVoffOutOfRange, 0, 0));
  }
  // transposed operand: element i of the contraction is row 8 (i / 4) + 4 hi + i % 4
  __device__ __forceinline__ void load_cols(float (&x)[16][FR<D>::DB], int b) const {
    const auto rs = rsrc(b);
    const int at = (4 * hi * (int)stride + c) * 4;
#pragma unroll
    for (int i = 0; i < 16; ++i)
#pragma unroll
      for (int db = 0; db < FR<D>::DB; ++db)
        x[i][db] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                                                 rs, 32 * db + c < cols ? at + 128 * db : kVoffOutOfRange,
                                                 (8 * (i / 4) + i % 4) * (int)stride * 4, 0));
  }
};

__device__ __forceinline__ void clear(f32x16& x) {
#pragma unroll
  for (int i = 0; i < 16; ++i) x[i] = 0.f;
}

// The 32 rows that the workgroup's waves share, as B operand: in LDS (in registers they would cost every
// wave D / 2 of them per tensor: the dK/dV kernel spilled 107 at D = 128), one 16-byte piece per four MFMAs.
template <int D>
__device__ __forceinline__ void stage_rows(float* lds, const float* rows, int64_t stride, int n, int cols, int tid) {
  constexpr int QPR = D / 4;
  const auto rs = wave_rsrc(rows, n > 0 ? ((n - 1) * (int)stride + cols) * 4 : 0);
#pragma unroll
  for (int e = tid; e < 32 * QPR; e += kWaves * 64) {
    const int r = e / QPR, col = (e % QPR) * 4;
    *reinterpret_cast<f32x4*>(lds + r * FR<D>::OSTR + col) = __builtin_bit_cast(
        f32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, col < cols ? r * (int)stride * 4 + col * 4 : kVoffOutOfRange, 0, 0));
  }
}
// Products over the head dim are summed 32 columns at a time: one chain over all of them left results of B2 H4 S128 D64
// 2.9e-7 (forward) and 4.3e-7 (gradients) off 64 bits, this 2.1e-7 and 3.7e-7 at the same speed (fa_f32.hip, whose waves
// hold 32 columns each: 2.6e-7 and 4.0e-7).
template <int D>
__device__ __forceinline__ f32x16 row_gemm_lds(const f32x4 (&a)[FR<D>::KJ], const float* b) {
  f32x16 s, t;
#pragma unroll
  for (int j = 0; j < FR<D>::KJ; ++j) {
    if (j % 4 == 0) clear(t);
    const f32x4 b4 = *reinterpret_cast<const f32x4*>(b + 8 * j);
#pragma unroll
    for (int e = 0; e < 4; ++e) t = mfma_f32(a[j][e], b4[e], t);
    if (j % 4 == 3) {
      s = j == 3 ? t : s + t;
      __builtin_amdgcn_sched_barrier(0);      // (no need for more pieces in flight)
    }
  }
  return s;
}
// one row of a tensor as a resident B operand
template <int D>
__device__ __forceinline__ void load_row(f32x4 (&x)[FR<D>::KJ], const float* row, int hi, int cols) {
#pragma unroll
  for (int j = 0; j < FR<D>::KJ; ++j)
    x[j] = 8 * j + 4 * hi < cols ? *reinterpret_cast<const f32x4*>(row + 8 * j + 4 * hi) : f32x4{0.f, 0.f, 0.f, 0.f};
}
template <int D>
__device__ __forceinline__ f32x16 row_gemm(const f32x4 (&a)[FR<D>::KJ], const f32x4 (&b)[FR<D>::KJ]) {
  f32x16 s, t;
#pragma unroll
  for (int j = 0; j < FR<D>::KJ; ++j) {
    if (j % 4 == 0) clear(t);
#pragma unroll
    for (int e = 0; e < 4; ++e) t = mfma_f32(a[j][e], b[j][e], t);
    if (j % 4 == 3) {
      s = j == 3 ? t : s + t;
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  return s;
}
template <int D>
__device__ __forceinline__ void col_gemm(const float (&a)[16][FR<D>::DB], const f32x16& x, f32x16 (&acc)[FR<D>::DB]) {
#pragma unroll
  for (int i = 0; i < 16; ++i)
#pragma unroll
    for (int db = 0; db < FR<D>::DB; ++db) acc[db] = mfma_f32(a[i][db], x[i], acc[db]);
}
template <int D>
__device__ __forceinline__ void zero(f32x16 (&acc)[FR<D>::DB]) {
#pragma unroll
  for (int db = 0; db < FR<D>::DB; ++db)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[db][i] = 0.f;
}
// a wave's 32 x D sums (transposed accumulators: a lane's row is lane % 32) to its LDS area
template <int D>
__device__ __forceinline__ void put(float* area, const f32x16 (&acc)[FR<D>::DB], int c, int hi) {
#pragma unroll
  for (int db = 0; db < FR<D>::DB; ++db)
#pragma unroll
    for (int g = 0; g < 4; ++g)
      *reinterpret_cast<f32x4*>(area + c * FR<D>::OSTR + 32 * db + 8 * g + 4 * hi) =
          f32x4{acc[db][4 * g], acc[db][4 * g + 1], acc[db][4 * g + 2], acc[db][4 * g + 3]};
}
// rows 0 .. n-1 of the four areas added up, times f, to rows of a tensor
template <int D>
__device__ __forceinline__ void sum_out(const float* areas, int n, float f, float* out, int64_t stride, int cols, int tid) {
  constexpr int QPR = D / 4;
  for (int e = tid; e < n * QPR; e += kWaves * 64) {
    const int r = e / QPR, col = (e % QPR) * 4;
    if (col >= cols) continue;
    f32x4 acc = *reinterpret_cast<const f32x4*>(areas + r * FR<D>::OSTR + col);
#pragma unroll
    for (int w = 1; w < kWaves; ++w) acc += *reinterpret_cast<const f32x4*>(areas + w * FR<D>::AREA + r * FR<D>::OSTR + col);
    *reinterpret_cast<f32x4*>(out + (int64_t)r * stride + col) = acc * f;
  }
}

// Work items in grid order: XCD x = id % 8 takes the x-th eighth of them, so that the items of a
// (sequence, kv-head) stay together (they read the same rows) and the XCDs have equal shares.
__device__ __forceinline__ int item_of(int id, int items) {
  const int chunk = (items + kNumXcd - 1) / kNumXcd, i = id / kNumXcd;
  const int item = (id % kNumXcd) * chunk + i;
  return i < chunk && item < items ? item : -1;
}

template <bool kWindowed>
__device__ __forceinline__ Window window_of(const MaskArgs& m, int sq, int sk) {
  Window w{0, 0};
  if (kWindowed) w = parse_window(m.causal_type, m.window_left, m.window_right, sq, sk);
  w.left = w.left > (1 << 30) ? (1 << 30) : (w.left < -(1 << 30) ? -(1 << 30) : w.left);
  w.right = w.right > (1 << 30) ? (1 << 30) : (w.right < -(1 << 30) ? -(1 << 30) : w.right);
  return w;
}

// Visible positions of a row as one range [lo, lo + rng]; `first` is added per element.
struct Range {
  int lo;
  bool none;
  unsigned rng;
  __device__ __forceinline__ Range(int l, int h, bool ok) : lo(l), none(!ok || h < l), rng(none ? 0u : (unsigned)(h - l)) {}
  __device__ __forceinline__ unsigned from(int n) const { return none ? 0x40000000u : (unsigned)(n - lo); }
};

template <int D, bool kWindowed, bool kBias, bool kDropout>
__global__ __launch_bounds__(256) void fwd_f32_rows_kernel(const FwdArgs a) {
  using C = FR<D>;
  extern __shared__ __attribute__((aligned(16))) char smem_raw[];
  float* areas = reinterpret_cast<float*>(smem_raw);
  float* ml = areas + kWaves * C::AREA;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63, c = lane & 31, hi = lane >> 5;
  const int nmt = (a.seq.max_seqlen_q + 31) / 32, group = a.hq / a.hk;
  if (kDropout && blockIdx.x == 0 && tid == 0) {
    uint64_t base = a.drop.offset2;      // modules/flash/kernel/fwd_kernel.py:199-207
    if (a.drop.offset1_ptr) base += *a.drop.offset1_ptr;
    if (a.seed_out) *a.seed_out = *a.drop.seed_ptr;
    if (a.offset_out) *a.offset_out = base;
  }
  const int item = item_of(blockIdx.x, a.num_zh * nmt);
  if (item < 0) return;
  // heads of a group next to each other, most visible keys (causal) first
  const int pair = item / (group * nmt), r = item % (group * nmt);
  const int z = pair / a.hk, hk = pair % a.hk, h = hk * group + r % group, mt = nmt - 1 - r / group;
  const SeqInfo si = get_seq(a.seq, z);
  const int q0 = mt * 32;
  if (q0 >= si.seqlen_q) return;
  const Window w = window_of<kWindowed>(a.mask, si.seqlen_q, si.seqlen_k);
  const BlockRanges br = block_ranges(kWindowed, w.left, w.right, q0, si.seqlen_q, si.seqlen_k, 32, 32);
  const int row = q0 + c, nrows = si.seqlen_q - q0 < 32 ? si.seqlen_q - q0 : 32;
  const int row_c = c < nrows ? row : si.seqlen_q - 1;

  f32x4 qreg[C::KJ];
  load_row<D>(qreg, reinterpret_cast<const float*>(a.q) + (int64_t)si.batch_index * a.sq.z + (int64_t)h * a.sq.h +
                        (int64_t)(si.q_start + row_c) * a.sq.s, hi, a.head_dim);
  const Block<D> K{reinterpret_cast<const float*>(a.k) + (int64_t)si.batch_index * a.sk.z + (int64_t)hk * a.sk.h +
                       (int64_t)si.k_start * a.sk.s, a.sk.s, si.seqlen_k, a.head_dim, c, hi};
  const Block<D> V{reinterpret_cast<const float*>(a.v) + (int64_t)si.batch_index * a.sv.z + (int64_t)hk * a.sv.h +
                       (int64_t)si.k_start * a.sv.s, a.sv.s, si.seqlen_k, a.head_dim_v, c, hi};
  const float* bptr = nullptr;
  if (kBias)
    bptr = reinterpret_cast<const float*>(a.bias) + (int64_t)si.batch_index * a.sb_z + (int64_t)h * a.sb_h + (int64_t)row_c * a.sb_m;
  DropoutState ds{};
  if (kDropout) ds = make_dropout(a.drop, z, h, a.hq, a.seq.max_seqlen_q, a.seq.max_seqlen_k);
  int m_lo = 0, m_hi = si.seqlen_k - 1;
  if (kWindowed) {
    m_lo = row - w.left > 0 ? row - w.left : 0;
    m_hi = row + w.right < m_hi ? row + w.right : m_hi;
  }
  const Range vis(m_lo, m_hi, true);
  const float qk_scale = a.sm_scale * kLog2e;
  const bool prescale = kBias || !(qk_scale > 0.f);      // as in fa_f32.hip
  const float sc = prescale ? 1.0f : qk_scale;

  f32x16 o[C::DB];
  zero<D>(o);
  float m_i = kNegBig, l_i = 0.f;
  f32x4 kr[C::KJ];
  float vc[16][C::DB];
  int j = br.lo + wave;
  if (j <= br.hi) K.load_rows(kr, j);
  for (; j <= br.hi; j += kWaves) {
    V.load_cols(vc, j);
    f32x16 s = row_gemm<D>(kr, qreg);
    phase();
    if (j + kWaves <= br.hi) K.load_rows(kr, j + kWaves);
    if (prescale) {
#pragma unroll
      for (int i = 0; i < 16; ++i) s[i] *= qk_scale;
    }
    if (kBias) {
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        int n = j * 32 + 8 * (i / 4) + 4 * hi + (i % 4);
        n = n < si.seqlen_k ? n : si.seqlen_k - 1;
        s[i] += bptr[(int64_t)n * a.sb_n] * kLog2e;   // fwd_kernel_inner.py:187
      }
    }
    if (!br.is_full(j)) {
      const unsigned d = vis.from(j * 32 + 4 * hi);
#pragma unroll
      for (int i = 0; i < 16; ++i) s[i] = d + (unsigned)(8 * (i / 4) + (i % 4)) <= vis.rng ? s[i] : -__builtin_inff();
    }
    float mx = s[0];
#pragma unroll
    for (int i = 1; i < 16; ++i) mx = fmaxf(mx, s[i]);
    const float m_new = fmaxf(m_i, cross_max(mx));
    const float alpha = fast_exp2((m_i - m_new) * sc);
    m_i = m_new;
    float rs = 0.f;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      s[i] = fast_exp2((s[i] - m_new) * sc);
      rs += s[i];                       // the row sum is over the undropped p (:213-214)
    }
    l_i = l_i * alpha + rs;
    if (__builtin_amdgcn_ballot_w64(alpha != 1.0f) != 0) {
#pragma unroll
      for (int db = 0; db < C::DB; ++db)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[db][i] *= alpha;
    }
    if (kDropout) {
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const uint32_t keep = dropout_keep4(ds, row, j * 32 + 8 * g + 4 * hi);
#pragma unroll
        for (int e = 0; e < 4; ++e) s[4 * g + e] = ((keep >> e) & 1u) ? s[4 * g + e] : 0.f;
      }
    }
    col_gemm<D>(vc, s, o);
    phase();
  }

  const float l = cross_sum(l_i);
  put<D>(areas + wave * C::AREA, o, c, hi);
  if (hi == 0) {
    ml[(wave * 32 + c) * 2] = m_i;
    ml[(wave * 32 + c) * 2 + 1] = l;
  }
  __syncthreads();
  constexpr int QPR = D / 4;
  float* out = reinterpret_cast<float*>(a.out) + (int64_t)si.batch_index * a.so.z + (int64_t)h * a.so.h + (int64_t)(si.q_start + q0) * a.so.s;
  for (int e = tid; e < nrows * QPR; e += 256) {
    const int rr = e / QPR, col = (e % QPR) * 4;
    float m = ml[rr * 2];
#pragma unroll
    for (int v = 1; v < kWaves; ++v) m = fmaxf(m, ml[(v * 32 + rr) * 2]);
    float lsum = 0.f;
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int v = 0; v < kWaves; ++v) {
      const float f = fast_exp2((ml[(v * 32 + rr) * 2] - m) * sc);
      lsum += f * ml[(v * 32 + rr) * 2 + 1];
      acc += f * *reinterpret_cast<const f32x4*>(areas + v * C::AREA + rr * C::OSTR + col);
    }
    const bool alive = lsum > 0.f;
    float inv = alive ? 1.0f / lsum : 0.f;
    if (kDropout) inv *= ds.scale;          // fwd_kernel.py:573-575
    if (col < a.head_dim_v) *reinterpret_cast<f32x4*>(out + (int64_t)rr * a.so.s + col) = acc * inv;
    if (a.lse && col == 0)
      a.lse[lse_offset(si, h, a.hq) + q0 + rr] = lse_of(m, sc, lsum);
  }
}

// dQ, dB and delta = rowsum(O dO) of its rows, which the dK/dV kernel reads (it runs after this one)
template <int D, bool kWindowed, bool kBias, bool kDropout>
__global__ __launch_bounds__(256, D <= 64 ? 2 : 1) void bwd_dq_f32_rows_kernel(const BwdArgs a) {
  using C = FR<D>;
  extern __shared__ __attribute__((aligned(16))) char smem_raw[];
  float* areas = reinterpret_cast<float*>(smem_raw);
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63, c = lane & 31, hi = lane >> 5;
  const int nmt = (a.seq.max_seqlen_q + 31) / 32, group = a.hq / a.hk;
  const int item = item_of(blockIdx.x, a.num_zh * nmt);
  if (item < 0) return;
  const int pair = item / (group * nmt), r = item % (group * nmt);
  const int z = pair / a.hk, hk = pair % a.hk, h = hk * group + r % group, mt = nmt - 1 - r / group;
  const SeqInfo si = get_seq(a.seq, z);
  const int q0 = mt * 32;
  if (q0 >= si.seqlen_q) return;
  const Window w = window_of<kWindowed>(a.mask, si.seqlen_q, si.seqlen_k);
  const BlockRanges br = block_ranges(kWindowed, w.left, w.right, q0, si.seqlen_q, si.seqlen_k, 32, 32);
  const int row = q0 + c, nrows = si.seqlen_q - q0 < 32 ? si.seqlen_q - q0 : 32;
  const bool row_ok = c < nrows;
  const int row_c = row_ok ? row : si.seqlen_q - 1;

  float *Qs = areas, *dOs = areas + C::AREA;
  stage_rows<D>(Qs, reinterpret_cast<const float*>(a.q) + (int64_t)si.batch_index * a.sq.z + (int64_t)h * a.sq.h +
                        (int64_t)(si.q_start + q0) * a.sq.s, a.sq.s, nrows, a.head_dim, tid);
  stage_rows<D>(dOs, reinterpret_cast<const float*>(a.dout) + (int64_t)si.batch_index * a.sdo.z + (int64_t)h * a.sdo.h +
                         (int64_t)(si.q_start + q0) * a.sdo.s, a.sdo.s, nrows, a.head_dim_v, tid);
  const float *q_b = Qs + c * C::OSTR + 4 * hi, *do_b = dOs + c * C::OSTR + 4 * hi;
  __syncthreads();
  float d_row = 0.f;
  {
    const float* op = reinterpret_cast<const float*>(a.out) + (int64_t)si.batch_index * a.so.z + (int64_t)h * a.so.h +
                      (int64_t)(si.q_start + row_c) * a.so.s;
#pragma unroll
    for (int j = 0; j < C::KJ; ++j) {
      if (8 * j + 4 * hi >= a.head_dim_v) continue;
      const f32x4 o4 = *reinterpret_cast<const f32x4*>(op + 8 * j + 4 * hi);
#pragma unroll
      for (int e = 0; e < 4; ++e) d_row += o4[e] * do_b[8 * j + e];
    }
    d_row = cross_sum(d_row);
    if (row_ok && hi == 0 && wave == 0) a.delta[lse_offset(si, h, a.hq) + row] = d_row;
  }
  const float l_row = a.lse[lse_offset(si, h, a.hq) + row_c] * kRcpLn2;               // bwd_kernel_dq.py:305
  const float qk_scale = a.sm_scale * kLog2e;
  const Block<D> K{reinterpret_cast<const float*>(a.k) + (int64_t)si.batch_index * a.sk.z + (int64_t)hk * a.sk.h +
                       (int64_t)si.k_start * a.sk.s, a.sk.s, si.seqlen_k, a.head_dim, c, hi};
  const Block<D> V{reinterpret_cast<const float*>(a.v) + (int64_t)si.batch_index * a.sv.z + (int64_t)hk * a.sv.h +
                       (int64_t)si.k_start * a.sv.s, a.sv.s, si.seqlen_k, a.head_dim_v, c, hi};
  const float* bptr = nullptr;
  if (kBias)
    bptr = reinterpret_cast<const float*>(a.bias) + (int64_t)si.batch_index * a.sb_z + (int64_t)h * a.sb_h + (int64_t)row_c * a.sb_m;
  const bool want_db = kBias && a.db != nullptr;
  float* dbhead = want_db ? reinterpret_cast<float*>(a.db) + (int64_t)si.batch_index * a.sdb_z + (int64_t)h * a.sdb_h : nullptr;
  float* dbptr = want_db ? dbhead + (int64_t)row_c * a.sdb_m : nullptr;
  DropoutState dst{};
  if (kDropout) dst = make_dropout(a.drop, z, h, a.hq, a.seq.max_seqlen_q, a.seq.max_seqlen_k);
  int m_lo = 0, m_hi = si.seqlen_k - 1;
  if (kWindowed) {
    m_lo = row - w.left > 0 ? row - w.left : 0;
    m_hi = row + w.right < m_hi ? row + w.right : m_hi;
  }
  const Range vis(m_lo, m_hi, true);

  f32x16 dq[C::DB];
  zero<D>(dq);
  f32x4 kr[C::KJ], vr[C::KJ];
  int j = br.lo + wave;
  if (j <= br.hi) { K.load_rows(kr, j); V.load_rows(vr, j); }
  for (; j <= br.hi; j += kWaves) {
    f32x16 s = row_gemm_lds<D>(kr, q_b);
    phase();
    float kc[16][C::DB];
    K.load_cols(kc, j);
    f32x16 dp = row_gemm_lds<D>(vr, do_b);
    phase();
    if (j + kWaves <= br.hi) V.load_rows(vr, j + kWaves);
    const bool masked = !br.is_full(j);
    const unsigned m_d = vis.from(j * 32 + 4 * hi);
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      uint32_t keep = 0xfu;
      if (kDropout) keep = dropout_keep4(dst, row, j * 32 + 8 * g + 4 * hi);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int i = 4 * g + e, n = j * 32 + 8 * g + 4 * hi + e;
        float x = s[i] * qk_scale - l_row;
        if (kBias) {
          const int nn = n < si.seqlen_k ? n : si.seqlen_k - 1;
          x = __builtin_fmaf(bptr[(int64_t)nn * a.sb_n], kLog2e, s[i] * qk_scale) - l_row;
        }
        if (masked) x = m_d + (unsigned)(8 * g + e) <= vis.rng ? x : -__builtin_inff();
        const float p = fast_exp2(x);
        float dpv = dp[i];
        if (kDropout) dpv = ((keep >> e) & 1u) ? dpv * dst.scale : 0.f;   // bwd_inner_dq.py:176-185
        s[i] = p * (dpv - d_row);
        if (want_db && row_ok && n < si.seqlen_k) dbptr[(int64_t)n * a.sdb_n] = s[i];   // :200-204
      }
    }
    col_gemm<D>(kc, s, dq);
    phase();
    if (j + kWaves <= br.hi) K.load_rows(kr, j + kWaves);
  }
  if (want_db) {
    // dB of key blocks that are never visited is zero: wave w sweeps the rows w, w + 4, ...
    for (int rr = wave; rr < nrows; rr += kWaves) {
      float* rowp = dbhead + (int64_t)(q0 + rr) * a.sdb_m;
      const int lo_end = br.lo <= br.hi ? br.lo * 32 : si.seqlen_k, hi_from = br.lo <= br.hi ? (br.hi + 1) * 32 : si.seqlen_k;
      for (int n = lane; n < lo_end && n < si.seqlen_k; n += 64) rowp[(int64_t)n * a.sdb_n] = 0.f;
      for (int n = hi_from + lane; n < si.seqlen_k; n += 64) rowp[(int64_t)n * a.sdb_n] = 0.f;
    }
  }
  __syncthreads();      // the operands' areas become the sums'
  put<D>(areas + wave * C::AREA, dq, c, hi);
  __syncthreads();
  sum_out<D>(areas, nrows, a.sm_scale, reinterpret_cast<float*>(a.dq) + (int64_t)si.batch_index * a.sdq.z + (int64_t)h * a.sdq.h +
                                           (int64_t)(si.q_start + q0) * a.sdq.s, a.sdq.s, a.head_dim, tid);
}

template <int D, bool kWindowed, bool kBias, bool kDropout>
__global__ __launch_bounds__(256, D <= 64 && !kDropout ? 2 : 1) void bwd_dkdv_f32_rows_kernel(const BwdArgs a) {
  using C = FR<D>;
  extern __shared__ __attribute__((aligned(16))) char smem_raw[];
  float* areas = reinterpret_cast<float*>(smem_raw);
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63, c = lane & 31, hi = lane >> 5;
  const int nnt = (a.seq.max_seqlen_k + 31) / 32, group = a.hq / a.hk;
  const int item = item_of(blockIdx.x, a.num_zh * nnt);      // (num_zh counts kv-heads here)
  if (item < 0) return;
  const int pair = item / nnt, nt = item % nnt;      // most visible queries (causal) first
  const int z = pair / a.hk, hk = pair % a.hk;
  const SeqInfo si = get_seq(a.seq, z);
  const int n0 = nt * 32;
  if (n0 >= si.seqlen_k) return;
  const Window w = window_of<kWindowed>(a.mask, si.seqlen_q, si.seqlen_k);
  // rows are keys here, columns are queries: key n sees query m iff n - right <= m <= n + left
  const BlockRanges br = block_ranges(kWindowed, w.right, w.left, n0, si.seqlen_k, si.seqlen_q, 32, 32);
  const int key = n0 + c, nkeys = si.seqlen_k - n0 < 32 ? si.seqlen_k - n0 : 32;
  const bool key_ok = c < nkeys;
  const int key_c = key_ok ? key : si.seqlen_k - 1;
  int q_lo = 0, q_hi = si.seqlen_q - 1;
  if (kWindowed) {
    q_lo = key - w.right > 0 ? key - w.right : 0;
    q_hi = key + w.left < q_hi ? key + w.left : q_hi;
  }
  const Range vis(q_lo, q_hi, key_ok);

  float *Ks = areas, *Vs = areas + C::AREA;
  stage_rows<D>(Ks, reinterpret_cast<const float*>(a.k) + (int64_t)si.batch_index * a.sk.z + (int64_t)hk * a.sk.h +
                        (int64_t)(si.k_start + n0) * a.sk.s, a.sk.s, nkeys, a.head_dim, tid);
  stage_rows<D>(Vs, reinterpret_cast<const float*>(a.v) + (int64_t)si.batch_index * a.sv.z + (int64_t)hk * a.sv.h +
                        (int64_t)(si.k_start + n0) * a.sv.s, a.sv.s, nkeys, a.head_dim_v, tid);
  const float *k_b = Ks + c * C::OSTR + 4 * hi, *v_b = Vs + c * C::OSTR + 4 * hi;
  __syncthreads();
  const float qk_scale = a.sm_scale * kLog2e;
  DropoutState drop0{};
  if (kDropout) drop0 = make_dropout_base(a.drop, a.seq.max_seqlen_k);

  f32x16 dk[C::DB], dv[C::DB];
  zero<D>(dk);
  zero<D>(dv);
  const int ntq = br.lo <= br.hi ? br.hi - br.lo + 1 : 0, total = group * ntq;
  auto q_of = [&](int it) {
    return Block<D>{reinterpret_cast<const float*>(a.q) + (int64_t)si.batch_index * a.sq.z + (int64_t)(hk * group + it / ntq) * a.sq.h +
                        (int64_t)si.q_start * a.sq.s, a.sq.s, si.seqlen_q, a.head_dim, c, hi};
  };
  auto do_of = [&](int it) {
    return Block<D>{reinterpret_cast<const float*>(a.dout) + (int64_t)si.batch_index * a.sdo.z + (int64_t)(hk * group + it / ntq) * a.sdo.h +
                        (int64_t)si.q_start * a.sdo.s, a.sdo.s, si.seqlen_q, a.head_dim_v, c, hi};
  };
  f32x4 qr[C::KJ], dor[C::KJ];
  int it = wave;
  if (it < total) { q_of(it).load_rows(qr, br.lo + it % ntq); do_of(it).load_rows(dor, br.lo + it % ntq); }
  for (; it < total; it += kWaves) {
    const int hq = hk * group + it / ntq, b = br.lo + it % ntq, m0 = b * 32;
    const Block<D> Q = q_of(it), dO = do_of(it);
    // L and delta of the block's rows, four at a time
    const int left = si.seqlen_q - m0 < 32 ? si.seqlen_q - m0 : 32;
    const auto lrs = wave_rsrc(a.lse + lse_offset(si, hq, a.hq) + m0, left * 4);
    const auto drs = wave_rsrc(a.delta + lse_offset(si, hq, a.hq) + m0, left * 4);
    f32x4 l4[4], d4[4];
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      l4[g] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(lrs, (8 * g + 4 * hi) * 4, 0, 0));
      d4[g] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(drs, (8 * g + 4 * hi) * 4, 0, 0));
    }
    f32x16 s = row_gemm_lds<D>(qr, k_b);
    phase();
    float qc[16][C::DB], dc[16][C::DB];
    dO.load_cols(dc, b);
    f32x16 dp = row_gemm_lds<D>(dor, v_b);
    phase();
    Q.load_cols(qc, b);
    DropoutState dst{};
    uint32_t kw[4];
    if (kDropout) {
      // one Philox call yields the bits of four consecutive keys, the lanes of a quad: quad lane q runs
      // the rows with m % 4 == q and hands the words round
      dst = dropout_for_head(drop0, z, hq, a.hq, a.seq.max_seqlen_q);
#pragma unroll
      for (int g = 0; g < 4; ++g) kw[g] = dropout_keep4(dst, m0 + 8 * g + 4 * hi + (lane & 3), key & ~3);
    }
    const float* bptr = nullptr;
    if (kBias)
      bptr = reinterpret_cast<const float*>(a.bias) + (int64_t)si.batch_index * a.sb_z + (int64_t)hq * a.sb_h + (int64_t)key_c * a.sb_n;
    const bool masked = !br.is_full(b);
    const unsigned q_d = vis.from(m0 + 4 * hi);
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int g = i / 4, e = i % 4;
      // p = exp2(s c + bias log2e - L log2e) (bwd_inner_dk_dv.py:187-188)
      const float l = l4[g][e] * kRcpLn2;
      float x = s[i] * qk_scale - l;
      if (kBias) {
        const int m = m0 + 8 * g + 4 * hi + e, mm = m < si.seqlen_q ? m : si.seqlen_q - 1;
        x = __builtin_fmaf(bptr[(int64_t)mm * a.sb_m], kLog2e, s[i] * qk_scale) - l;
      }
      if (masked) x = q_d + (unsigned)(8 * g + e) <= vis.rng ? x : -__builtin_inff();
      const float p = fast_exp2(x);
      float pv = p, dpv = dp[i];
      if (kDropout) {
        int w4;
        switch (e) {       // quad_perm: [e, e, e, e]
          case 0: w4 = __builtin_amdgcn_mov_dpp((int)kw[g], 0x00, 0xf, 0xf, true); break;
          case 1: w4 = __builtin_amdgcn_mov_dpp((int)kw[g], 0x55, 0xf, 0xf, true); break;
          case 2: w4 = __builtin_amdgcn_mov_dpp((int)kw[g], 0xaa, 0xf, 0xf, true); break;
          default: w4 = __builtin_amdgcn_mov_dpp((int)kw[g], 0xff, 0xf, 0xf, true); break;
        }
        const bool keep = ((uint32_t)w4 >> (lane & 3)) & 1u;
        pv = keep ? p * dst.scale : 0.f;                       // :200-201
        dpv = keep ? dpv * dst.scale : 0.f;                    // :239-240
      }
      s[i] = pv;                                               // p as the dV GEMM sees it (dropped and scaled)
      dp[i] = p * (dpv - d4[g][e]);                            // dS uses the undropped p (:242)
    }
    col_gemm<D>(dc, s, dv);
    phase();
    if (it + kWaves < total) q_of(it + kWaves).load_rows(qr, br.lo + (it + kWaves) % ntq);
    col_gemm<D>(qc, dp, dk);
    phase();
    if (it + kWaves < total) do_of(it + kWaves).load_rows(dor, br.lo + (it + kWaves) % ntq);
  }

  __syncthreads();      // the operands' areas become the sums'
  put<D>(areas + wave * C::AREA, dk, c, hi);
  __syncthreads();
  sum_out<D>(areas, nkeys, a.sm_scale, reinterpret_cast<float*>(a.dk) + (int64_t)si.batch_index * a.sdk.z + (int64_t)hk * a.sdk.h +
                                           (int64_t)(si.k_start + n0) * a.sdk.s, a.sdk.s, a.head_dim, tid);      // bwd_kernel_dk_dv.py:387-389
  __syncthreads();
  put<D>(areas + wave * C::AREA, dv, c, hi);
  __syncthreads();
  sum_out<D>(areas, nkeys, 1.0f, reinterpret_cast<float*>(a.dv) + (int64_t)si.batch_index * a.sdv.z + (int64_t)hk * a.sdv.h +
                                     (int64_t)(si.k_start + n0) * a.sdv.s, a.sdv.s, a.head_dim_v, tid);
}

template <auto kern, int smem, typename Args>
hipError_t launch(int items, hipStream_t stream, const Args& a) {
  if (items == 0) return hipSuccess;   // an empty tensor: nothing to write
  if (smem > 64 * 1024) {
    static std::atomic<uint64_t> lds_set{0};
    hipError_t e = allow_large_lds(reinterpret_cast<const void*>(kern), smem, lds_set);
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL(kern, dim3((unsigned)(kNumXcd * ((items + kNumXcd - 1) / kNumXcd))), dim3(256), smem, stream, a);
  return hipGetLastError();
}

#define FA_F32_SWITCH(CALL)                                            \
  switch ((windowed ? 4 : 0) | (bias ? 2 : 0) | (dropout ? 1 : 0)) {   \
    case 0: return CALL(false, false, false);                          \
    case 1: return CALL(false, false, true);                           \
    case 2: return CALL(false, true, false);                           \
    case 3: return CALL(false, true, true);                            \
    case 4: return CALL(true, false, false);                           \
    case 5: return CALL(true, false, true);                            \
    case 6: return CALL(true, true, false);                            \
    default: return CALL(true, true, true);                            \
  }

template <int D>
hipError_t run_fwd_d(const FwdArgs& a0, bool windowed, bool bias, bool dropout, hipStream_t s) {
  FwdArgs a = a0;
  a.num_zh = nseq_of(a.seq, a.batch) * a.hq;
  const int items = a.num_zh * ((a.seq.max_seqlen_q + 31) / 32);
#define FA_CALL(W, B, P) launch<fwd_f32_rows_kernel<D, W, B, P>, FR<D>::SMEM>(items, s, a)
  FA_F32_SWITCH(FA_CALL)
#undef FA_CALL
}

template <int D>
hipError_t run_bwd_d(int kernel_slot, const BwdArgs& a0, bool windowed, bool bias, bool dropout, hipStream_t s) {
  BwdArgs a = a0;
  if (kernel_slot == 1) {
    a.num_zh = nseq_of(a.seq, a.batch) * a.hk;
    const int items = a.num_zh * ((a.seq.max_seqlen_k + 31) / 32);
#define FA_CALL(W, B, P) launch<bwd_dkdv_f32_rows_kernel<D, W, B, P>, FR<D>::SMEM>(items, s, a)
    FA_F32_SWITCH(FA_CALL)
#undef FA_CALL
  }
  a.num_zh = nseq_of(a.seq, a.batch) * a.hq;
  const int items = a.num_zh * ((a.seq.max_seqlen_q + 31) / 32);
#define FA_CALL(W, B, P) launch<bwd_dq_f32_rows_kernel<D, W, B, P>, FR<D>::SMEM>(items, s, a)
  FA_F32_SWITCH(FA_CALL)
#undef FA_CALL
}

}  // namespace

TileShape f32_rows_tile_shape(int head_dim) {
  return TileShape{32, 32, kWaves, head_dim <= 64 ? FR<64>::SMEM : FR<128>::SMEM};
}
hipError_t run_fwd_f32_rows(int head_dim, const FwdArgs& a, bool windowed, bool bias, bool dropout, hipStream_t s) {
  return head_dim <= 64 ? run_fwd_d<64>(a, windowed, bias, dropout, s) : run_fwd_d<128>(a, windowed, bias, dropout, s);
}
hipError_t run_bwd_f32_rows(int head_dim, int kernel_slot, const BwdArgs& a, bool windowed, bool bias, bool dropout, hipStream_t s) {
  return head_dim <= 64 ? run_bwd_d<64>(kernel_slot, a, windowed, bias, dropout, s)
                        : run_bwd_d<128>(kernel_slot, a, windowed, bias, dropout, s);
}

}  // namespace fa
