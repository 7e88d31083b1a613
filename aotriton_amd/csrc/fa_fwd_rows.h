// Forward for few query rows per K/V head (decode, short prompt chunks): gfx950, MFMA 32x32x16.
//
// The tile of fwd_kernel is 256 (128 at D = 256) query rows of ONE q-head.  With one query per
// sequence it has one row to work on, the q-heads of a GQA group each stream the same K/V, and a
// (batch, head) pair has one workgroup however long the keys are.  Here a work item is
//   32 packed rows = (query, q-head of the group) pairs of one K/V head, row r = query * group + head
//   x one of `splits` parts of the visible keys,
// so K/V are read once per group and the keys of a pair are spread over many workgroups.  The four
// waves of a workgroup take blocks of 32 keys in turn, each with its own online softmax; the waves
// meet once at the end (LDS), the splits in a second kernel (combine_rows_kernel, fp32 partial sums
// in scratch memory).
//
// What bounds it: HBM (one query per sequence: 1 FLOP per byte and row).  Hence no shared tiles and no
// barrier in the loop: the K operand of S^T = K Q^T is loaded from global memory as it lies (row =
// lane % 32, 16 bytes of it), V passes through a wave-private LDS area because O^T = V^T P^T needs it
// transposed, and the next block's loads are issued as soon as the registers of this one are free.
// With two workgroups per CU up to 8 x 16 KB (D = 128) are in flight per CU; 48 KB are what the latency
// times the HBM rate asks for.  More than 32 rows only re-read K/V from L2 (the row blocks of a part run
// on one XCD, next to each other).
#pragma once
#include "fa_combine.h"
#include "fa_device.h"

namespace fa {

constexpr int kRowsBlock = 32;      // packed rows per item, keys per step of a wave
constexpr int kRowsWaves = 4;

template <int D>
struct RowsSmem {
  static constexpr int VSTR = D + 32;                    // elements; +64 B per row: transposing reads sweep all banks
  static constexpr int V_BYTES = 32 * VSTR * 2;          // per wave
  static constexpr int OSTR = D + 4;                     // floats per row of a wave's partial O
  static constexpr int O_BYTES = 32 * OSTR * 4;          // per wave
  static constexpr int ML_OFF = kRowsWaves * (V_BYTES > O_BYTES ? V_BYTES : O_BYTES);
  static constexpr int BYTES = ML_OFF + kRowsWaves * 32 * 8;
};

// kMask: the bias is FwdArgs::key_mask's.  (As a case at run time it cost a bias 1-5 %: kernel time of B1 H12 S512 D64 fp16 causal
// 9.2 us, now 8.8-9.0.)
template <typename T, int D, bool kWindowed, bool kBias, bool kPad, bool kMask>
__global__ __attribute__((amdgpu_flat_work_group_size(256, 256)))
__attribute__((amdgpu_waves_per_eu(D <= 128 ? 2 : 1, D <= 128 ? 2 : 1)))
void fwd_rows_kernel(const FwdArgs a) {
  extern __shared__ __attribute__((aligned(16))) char smem_raw[];
  using Tr = Traits<T>;
  using op_t = typename Tr::op_t;
  using q4_t = typename Tr::q4_t;
  using SM = RowsSmem<D>;
  constexpr int KS = D / 16, DB = D / 32;
  constexpr int VSTR = SM::VSTR, OSTR = SM::OSTR;
  constexpr int LPR = D / 8, RPI = 64 / LPR, CHV = 32 / RPI;      // V: lanes per row, rows per access, accesses

  // units (pair, split) go round the XCDs, the row blocks of a unit follow each other on one
  const int xcd = blockIdx.x % kNumXcd, idx = blockIdx.x / kNumXcd;
  const int unit = (idx / a.row_blocks) * kNumXcd + xcd, rb = idx % a.row_blocks;
  const int pair = unit / a.splits, split = unit % a.splits;
  const int group = a.hq / a.hk;
  if (pair * group >= a.num_zh) return;
  const int z = pair / a.hk, hk = pair % a.hk;
  const SeqInfo si = get_seq(a.seq, z);
  const int rows = si.seqlen_q * group;
  const int r0 = rb * kRowsBlock;
  if (r0 >= rows) return;
  const int nrows = rows - r0 < kRowsBlock ? rows - r0 : kRowsBlock;

  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63, c = lane & 31, hi = lane >> 5;
  const int d_qk = kPad ? a.head_dim : D, d_v = kPad ? a.head_dim_v : D;

  // this lane's packed row
  const bool row_ok = c < nrows;
  const int pr = r0 + (row_ok ? c : nrows - 1);
  const int row = pr / group, h = hk * group + pr % group;
  const int row_first = r0 / group, row_last = (r0 + nrows - 1) / group;

  // visible keys: of the block (all its rows together) and of this lane's row
  Window w{0, 0};
  if (kWindowed) w = parse_window(a.mask.causal_type, a.mask.window_left, a.mask.window_right, si.seqlen_q, si.seqlen_k);
  w.left = w.left > (1 << 30) ? (1 << 30) : (w.left < -(1 << 30) ? -(1 << 30) : w.left);
  w.right = w.right > (1 << 30) ? (1 << 30) : (w.right < -(1 << 30) ? -(1 << 30) : w.right);
  int key_lo = 0, key_hi = si.seqlen_k - 1, m_lo = 0, m_hi = si.seqlen_k - 1;
  int all_lo = 0, all_hi = si.seqlen_k - 1;      // keys that every row of the block sees
  if (kWindowed) {
    key_lo = row_first - w.left > 0 ? row_first - w.left : 0;
    key_hi = row_last + w.right < key_hi ? row_last + w.right : key_hi;
    m_lo = row - w.left > 0 ? row - w.left : 0;
    m_hi = row + w.right < m_hi ? row + w.right : m_hi;
    all_lo = row_last - w.left > 0 ? row_last - w.left : 0;
    all_hi = row_first + w.right < all_hi ? row_first + w.right : all_hi;
  }
  const bool m_none = m_hi < m_lo;
  const unsigned m_rng = m_none ? 0u : (unsigned)(m_hi - m_lo);
  const int blk_lo = key_lo / 32, blk_n = key_hi >= key_lo ? key_hi / 32 - blk_lo + 1 : 0;
  const int per = (blk_n + a.splits - 1) / a.splits;
  const int b0 = blk_lo + split * per;
  const int b1 = (split + 1) * per < blk_n ? b0 + per : blk_lo + blk_n;      // (b1 <= b0: nothing to do)

  // ---- Q rows as the B operand (col = packed row), straight from global memory ----------------
  op_t qreg[KS];
  {
    const T* qp = reinterpret_cast<const T*>(a.q) + (int64_t)si.batch_index * a.sq.z + (int64_t)h * a.sq.h +
                  (int64_t)(si.q_start + row) * a.sq.s + 8 * hi;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      qreg[ks] = op_t{};
      if (row_ok && (!kPad || 16 * ks + 8 * hi < d_qk)) qreg[ks] = *reinterpret_cast<const op_t*>(qp + 16 * ks);
    }
  }

  const T* kbase = reinterpret_cast<const T*>(a.k) + (int64_t)si.batch_index * a.sk.z + (int64_t)hk * a.sk.h +
                   (int64_t)si.k_start * a.sk.s;
  const T* vbase = reinterpret_cast<const T*>(a.v) + (int64_t)si.batch_index * a.sv.z + (int64_t)hk * a.sv.h +
                   (int64_t)si.k_start * a.sv.s;
  const T* bptr = nullptr;
  const uint8_t* mptr = nullptr;      // kMask
  if (kBias) {
    const int64_t at = (int64_t)si.batch_index * a.sb_z + (int64_t)h * a.sb_h + (int64_t)row * a.sb_m;
    bptr = reinterpret_cast<const T*>(a.bias) + at;
    mptr = reinterpret_cast<const uint8_t*>(a.bias) + at;
  }
  const bool bias_vec = kBias && a.sb_n == 1 && ((a.sb_m | a.sb_h | a.sb_z) & 3) == 0 &&
                        (reinterpret_cast<uintptr_t>(a.bias) & 7) == 0;

  const int k_row = (int)a.sk.s * 2, v_row = (int)a.sv.s * 2;
  const int kvoff = c * k_row + 16 * hi;
  const int vr0 = lane / LPR, vc0 = lane % LPR;
  const int vvoff = !kPad || vc0 * 8 < d_v ? vr0 * v_row + vc0 * 16 : kVoffOutOfRange;
  op_t kreg[KS], vreg[CHV];
  // rows past the end of the keys and columns past the head dim read as zero
  auto load_block = [&](int b) {
    const int left = si.seqlen_k - b * 32;
    const int n = left < 32 ? left : 32;
    const auto krs = wave_rsrc(kbase + (int64_t)b * 32 * a.sk.s, n > 0 ? (n - 1) * k_row + d_qk * 2 : 0);
    const auto vrs = wave_rsrc(vbase + (int64_t)b * 32 * a.sv.s, n > 0 ? (n - 1) * v_row + d_v * 2 : 0);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const int off = !kPad || 16 * ks + 8 * hi < d_qk ? kvoff + 32 * ks : kVoffOutOfRange;
      kreg[ks] = __builtin_bit_cast(op_t, __builtin_amdgcn_raw_buffer_load_b128(krs, off, 0, 0));
    }
#pragma unroll
    for (int i = 0; i < CHV; ++i)
      vreg[i] = __builtin_bit_cast(op_t, __builtin_amdgcn_raw_buffer_load_b128(vrs, vvoff, i * RPI * v_row, 0));
  };

  T* vs = reinterpret_cast<T*>(smem_raw + wave * SM::V_BYTES);
  const int v_st = vr0 * VSTR + vc0 * 8;
  const T* v_ld = vs + (4 * hi + (lane & 15) / 4) * VSTR + 16 * ((lane >> 4) & 1) + 4 * (lane & 3);      // see lds_read_tr8

  f32x16 o[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[db][i] = 0.f;
  float m_i = kNegBig, l_i = 0.f;      // running maximum (units of s below); this lane's half of the row sum
  const float qk_scale = a.sm_scale * kLog2e;
  const bool prescale = kBias || !(qk_scale > 0.f);      // as in fwd_item
  const float sc = prescale ? 1.0f : qk_scale;

  int b = b0 + wave;
  if (b < b1) load_block(b);
  for (; b < b1; b += kRowsWaves) {
    f32x16 s;
#pragma unroll
    for (int i = 0; i < 16; ++i) s[i] = 0.f;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) s = Tr::mfma(kreg[ks], qreg[ks], s);
#pragma unroll
    for (int i = 0; i < CHV; ++i) *reinterpret_cast<op_t*>(vs + v_st + i * RPI * VSTR) = vreg[i];
    if (b + kRowsWaves < b1) load_block(b + kRowsWaves);

    if (prescale)
#pragma unroll
      for (int i = 0; i < 16; ++i) s[i] *= qk_scale;
    const int n0 = b * 32;
    if (kMask) {
      // (0 or -inf is added, not selected: what an additive mask makes of inf and NaN)
      if (a.sb_n == 1 && n0 + 32 <= si.seqlen_k) {
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          uint32_t m4;
          __builtin_memcpy(&m4, mptr + n0 + 8 * g + 4 * hi, 4);      // (masks may start anywhere)
#pragma unroll
          for (int r = 0; r < 4; ++r) s[4 * g + r] += (m4 & 0xffu << 8 * r) != 0 ? 0.f : -__builtin_inff();
        }
      } else {
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          int n = n0 + 8 * (i / 4) + 4 * hi + (i % 4);
          n = n < si.seqlen_k ? n : si.seqlen_k - 1;
          s[i] += mptr[(int64_t)n * a.sb_n] != 0 ? 0.f : -__builtin_inff();
        }
      }
    } else if (kBias) {
      if (bias_vec && n0 + 32 <= si.seqlen_k) {
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const q4_t b4 = *reinterpret_cast<const q4_t*>(bptr + n0 + 8 * g + 4 * hi);
#pragma unroll
          for (int r = 0; r < 4; ++r) s[4 * g + r] += (float)b4[r] * kLog2e;
        }
      } else {
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          int n = n0 + 8 * (i / 4) + 4 * hi + (i % 4);
          n = n < si.seqlen_k ? n : si.seqlen_k - 1;
          s[i] += (float)bptr[(int64_t)n * a.sb_n] * kLog2e;
        }
      }
    }
    if (n0 < all_lo || n0 + 31 > all_hi) {
      // column n is visible iff m_lo <= n <= m_hi: one unsigned comparison (an empty range fails every element)
      const unsigned d = m_none ? 0x40000000u : (unsigned)(n0 + 4 * hi - m_lo);
#pragma unroll
      for (int i = 0; i < 16; ++i) s[i] = d + (unsigned)(8 * (i / 4) + (i % 4)) <= m_rng ? s[i] : -__builtin_inff();
    }

    float mx = s[0];
#pragma unroll
    for (int i = 1; i < 16; ++i) mx = fmaxf(mx, s[i]);
    mx = cross_max(mx);
    // lazy rescaling and exp2 on differences, as in fwd_item
    const float m_cand = fmaxf(m_i, mx);
    const bool upd = (m_cand - m_i) * sc > 8.0f;
    const float m_new = upd ? m_cand : m_i;
    const float alpha = fast_exp2((m_i - m_new) * sc);
    m_i = m_new;
    float rs = 0.f;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      s[i] = fast_exp2((s[i] - m_new) * sc);
      rs += s[i];
    }
    l_i = l_i * alpha + rs;
    if (__builtin_amdgcn_ballot_w64(upd) != 0) {
#pragma unroll
      for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[db][i] *= alpha;
    }
    const op_t p0 = pack8<T>(s, 0), p1 = pack8<T>(s, 1);
#pragma unroll
    for (int db = 0; db < DB; ++db) o[db] = Tr::mfma(lds_read_tr8<T>(v_ld + db * 32, VSTR), p0, o[db]);
#pragma unroll
    for (int db = 0; db < DB; ++db) o[db] = Tr::mfma(lds_read_tr8<T>(v_ld + 16 * VSTR + db * 32, VSTR), p1, o[db]);
  }

  // ---- the four waves' partial results meet in LDS --------------------------------------------
  const float l = cross_sum(l_i);
  __syncthreads();      // the V areas become the O areas
  float* ml = reinterpret_cast<float*>(smem_raw + SM::ML_OFF);
  float* ow = reinterpret_cast<float*>(smem_raw + wave * SM::O_BYTES);
  if (row_ok) {
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int g = 0; g < 4; ++g)
        *reinterpret_cast<f32x4*>(ow + c * OSTR + 32 * db + 8 * g + 4 * hi) =
            f32x4{o[db][4 * g], o[db][4 * g + 1], o[db][4 * g + 2], o[db][4 * g + 3]};
    if (hi == 0) {
      ml[(wave * 32 + c) * 2] = m_i;      // (kNegBig where the wave saw no key of the row; l is 0 then)
      ml[(wave * 32 + c) * 2 + 1] = l;
    }
  }
  __syncthreads();
  constexpr int QPR = D / 4;      // pieces of four columns per row
  for (int e = tid; e < nrows * QPR; e += 256) {
    const int r = e / QPR, col = (e % QPR) * 4;
    float m = ml[r * 2];
#pragma unroll
    for (int v = 1; v < kRowsWaves; ++v) m = fmaxf(m, ml[(v * 32 + r) * 2]);
    float lsum = 0.f;
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int v = 0; v < kRowsWaves; ++v) {
      const float f = fast_exp2((ml[(v * 32 + r) * 2] - m) * sc);
      lsum += f * ml[(v * 32 + r) * 2 + 1];
      acc += f * *reinterpret_cast<const f32x4*>(smem_raw + v * SM::O_BYTES + (r * OSTR + col) * 4);
    }
    if (a.splits > 1) {
      const int64_t part = ((int64_t)(pair * a.row_blocks + rb) * a.splits + split) * a.part_rows + r;
      *reinterpret_cast<f32x4*>(a.part_o + part * D + col) = acc;
      if (col == 0) {
        a.part_ml[part * 2] = m;
        a.part_ml[part * 2 + 1] = lsum;
      }
    } else if (col < d_v) {
      const int pq = (r0 + r) / group, ph = hk * group + (r0 + r) % group;
      const bool alive = lsum > 0.f;
      const float inv = alive ? 1.0f / lsum : 0.f;
      q4_t t4;
#pragma unroll
      for (int i = 0; i < 4; ++i) t4[i] = Tr::cvt(acc[i] * inv);
      *reinterpret_cast<q4_t*>(reinterpret_cast<T*>(a.out) + (int64_t)si.batch_index * a.so.z + (int64_t)ph * a.so.h +
                               (int64_t)(si.q_start + pq) * a.so.s + col) = t4;
      if (a.lse && col == 0)
        a.lse[lse_offset(si, ph, a.hq) + pq] = lse_of(m, sc, lsum);
    }
  }
}

template <typename T, int D, bool kWindowed, bool kBias, bool kPad, bool kMask = false>
hipError_t launch_fwd_rows_variant(const FwdArgs& a, hipStream_t stream) {
  auto kern = fwd_rows_kernel<T, D, kWindowed, kBias, kPad, kMask>;
  constexpr int smem = RowsSmem<D>::BYTES;
  if (smem > 64 * 1024) {
    static std::atomic<uint64_t> lds_set{0};
    const hipError_t e = allow_large_lds(reinterpret_cast<const void*>(kern), smem, lds_set);
    if (e != hipSuccess) return e;
  }
  const int pairs = a.num_zh / a.hq * a.hk;
  const int units = (pairs * a.splits + kNumXcd - 1) / kNumXcd;
  if (units == 0 || a.row_blocks == 0) return hipSuccess;
  hipLaunchKernelGGL(kern, dim3((unsigned)(kNumXcd * units * a.row_blocks)), dim3(256), smem, stream, a);
  hipError_t e = hipGetLastError();
  if (e == hipSuccess && a.splits > 1) e = launch_combine_rows<T, D>(a, pairs, stream);
  return e;
}

// a.row_blocks, a.splits, a.part_rows and the scratch pointers are the caller's
template <typename T, int D, bool kPad>
hipError_t launch_fwd_rows(const FwdArgs& a, bool windowed, bool bias, hipStream_t stream) {
  FwdArgs b = a;
  b.num_zh = nseq_of(a.seq, a.batch) * a.hq;
  b.part_group = a.hq / a.hk;
  b.part_block = kRowsBlock;
  if constexpr (D <= 128)      // (the library takes no key mask above)
    if (b.key_mask)
      return windowed ? launch_fwd_rows_variant<T, D, true, true, kPad, true>(b, stream)
                      : launch_fwd_rows_variant<T, D, false, true, kPad, true>(b, stream);
  switch ((windowed ? 2 : 0) | (bias ? 1 : 0)) {
    case 0: return launch_fwd_rows_variant<T, D, false, false, kPad>(b, stream);
    case 1: return launch_fwd_rows_variant<T, D, false, true, kPad>(b, stream);
    case 2: return launch_fwd_rows_variant<T, D, true, false, kPad>(b, stream);
    default: return launch_fwd_rows_variant<T, D, true, true, kPad>(b, stream);
  }
}

}  // namespace fa
