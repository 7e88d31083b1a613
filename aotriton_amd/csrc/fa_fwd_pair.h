// Forward work item of 256 columns: 128 query rows on eight waves, two per SIMD, that share 32 rows by product.
//
// Same arithmetic as fwd_item (fa_fwd_impl.h; modules/flash/kernel/fwd_kernel.py:83-644, fwd_kernel_inner.py:46-287 of the
// reference), other division of the work:
//   wave w      S^T(u) = K(u) Q^T, the online softmax of unit u - 1 (bias, mask, row maximum, row sum) behind it    holds Q
//   wave w + 4  O^T += V(u - 2)^T P(u - 2)^T; requests K and V                                                      holds O
// P goes from one to the other through LDS as the operand it becomes, with the factor that takes O to the rows' new reference
// where it has moved.
//
// Why: at 256 columns the accumulators of 32 rows take 128 registers and their Q rows 64; a wave with both runs alone on its SIMD, and
// its MFMAs, the vector work of its softmax and its LDS traffic are issued one after the other.  Apart, each half fits 256 registers.
//
// A step is 32 keys and has one barrier: in the time between two of them the first waves work on unit u and the second ones on
// unit u - 2.  K and V go straight into LDS (swizzled; three stages each), two steps ahead of their use.  A CU takes 16 cycles for each
// load into LDS, so the eight of a wave stand between its MFMAs: in front of them they held it up for 650 cycles of a step's 2300.
//
// Bound: the two waves' 32 MFMAs take 1024 cycles of a step's 1950 (at 1.9 GHz); what is left is that after the barrier both wait for their first
// operands and before it for the last exponentials and P, with the matrix pipe idle.  With dropout the rounds of a unit's Philox calls (300 cycles
// each next to the other wave) are longer than that: with all four in the second wave its step takes 2800 and the first one's 2000; two each, us, window
// S1801 38.5 -> 37.4, S8192 571 -> 562 (one card; long calls run at the clock that the power leaves, and moving work between the waves gives them less).
// Level or slower: more operands in flight, wave priorities, the first operands of the next unit read in front of the barrier (a stage
// more of K), the second waves over 64 columns of all rows (less LDS traffic, 5-8 % slower), the first product of Philox round 2, which the counter's upper
// word alone decides, kept along a row (19 registers more; S8192 529 -> 525, S4096 causal 365 -> 373).
//
// Measured, us, one wave per SIMD with all of it interleaved -> this, one card: B2 H16 S8192 fp16 window 1024, bias and dropout 618 -> 530, B1 H8 S1801
// 52 -> 38; B2 H16 S4096 with a bias 728 -> 576 (755 -> 955 TFLOP/s); B1 H16 Hk4 S8192 bf16 causal 716 -> 576, B2 S2048 96 -> 77.
#pragma once
#include <type_traits>

#include "fa_device.h"
#include "fa_wide.h"

namespace fa {

struct FwdPairSmem {
  static constexpr int D = 256, BN = 32, STAGES = 3;
  static constexpr int TILE_BYTES = BN * D * 2;
  static constexpr int V_OFF = STAGES * TILE_BYTES;
  static constexpr int P_OFF = 2 * V_OFF, P_BYTES = 4 * 2048;            // per step: two operands per lane of the four first waves
  static constexpr int FACTOR_OFF = P_OFF + 2 * P_BYTES;                 // and a float
  static constexpr int KEEP_OFF = FACTOR_OFF + 2 * 1024;                 // keep bits, a word per lane of the four first waves
  static constexpr int BIAS_OFF = KEEP_OFF + 2 * 1024, BIAS_ROW = 64 + 16, BIAS_BYTES = 32 * BIAS_ROW;      // per first wave, for units in turn
  static constexpr int BYTES = BIAS_OFF + 2 * 4 * BIAS_BYTES;
  static constexpr int ROW_STR = D * 2 + 16;                             // O rows on their way out, where K and V were
  static_assert(4 * 32 * ROW_STR <= P_OFF, "four waves' rows");
  static_assert(TILE_BYTES % kSwzAlign == 0 && V_OFF % kSwzAlign == 0, "stages leave the swizzled bits of an address alone");
};

template <typename T, bool kWindowed, bool kBias, bool kDropout, int kPad>
__device__ __forceinline__ void fwd_item_pair(const FwdArgs& a, const int z, const int h, const int mt, char* smem_raw) {
  using Tr = Traits<T>;
  using op_t = typename Tr::op_t;
  using q4_t = typename Tr::q4_t;
  using SM = FwdPairSmem;
  constexpr int D = SM::D, BN = SM::BN, BM = 128;
  constexpr int KS = D / 16, DB = D / 32, ROWB = Swz<D>::ROWB;

  const int lane = threadIdx.x & 63, c = lane & 31, hi = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int w = wave & 3;                        // row block
  const bool first = wave < 4;
  const int d_qk = kPad ? a.head_dim : D, d_v = kPad ? a.head_dim_v : D;

  const SeqInfo si = uniform(get_seq(a.seq, z));
  const int q0 = mt * BM;
  if (q0 >= si.seqlen_q) return;

  Window win{0, 0};
  if (kWindowed) win = parse_window(a.mask.causal_type, a.mask.window_left, a.mask.window_right, si.seqlen_q, si.seqlen_k);
  // keep row +/- window inside int32
  win.left = win.left > (1 << 30) ? (1 << 30) : (win.left < -(1 << 30) ? -(1 << 30) : win.left);
  win.right = win.right > (1 << 30) ? (1 << 30) : (win.right < -(1 << 30) ? -(1 << 30) : win.right);
  const BlockRanges br = block_ranges(kWindowed, win.left, win.right, q0, si.seqlen_q, si.seqlen_k, BM, BN);

  const int hk = h / (a.hq / a.hk);                       // fwd_kernel.py:360
  const int w_rmin = q0 + w * 32;                         // first row of the block
  const int wrows = si.seqlen_q - w_rmin < 32 ? si.seqlen_q - w_rmin : 32;   // valid rows, may be <= 0
  const int w_rmax = w_rmin + (wrows > 0 ? wrows : 1) - 1;
  const int row = w_rmin + c;                             // this lane's row
  const bool row_ok = row < si.seqlen_q;
  const int smem0 = lds_offset(smem_raw);

  auto store_rows = [&](bool zeros) {
    // whole rows of Out: 16 bytes per lane, consecutive lanes along a row
    constexpr int LPRQ = D / 8, RPQ = 64 / LPRQ;
    const int rq = lane / LPRQ, cq = lane % LPRQ;
    T* ow = reinterpret_cast<T*>(a.out) + (int64_t)si.batch_index * a.so.z + (int64_t)h * a.so.h + (int64_t)(si.q_start + w_rmin) * a.so.s;
    const auto ors = wave_rsrc(ow, wrows > 0 ? ((wrows - 1) * (int)a.so.s + d_v) * 2 : 0);
    const int ovoff = cq * 8 < d_v ? rq * (int)a.so.s * 2 + cq * 16 : kVoffOutOfRange;
    const int at = smem0 + w * 32 * SM::ROW_STR + rq * SM::ROW_STR + cq * 16;
#pragma unroll
    for (int i = 0; i < 32 / RPQ; ++i) {
      u32x4_t x = {0u, 0u, 0u, 0u};
      if (!zeros) x = lds_read<u32x4_t>(at + i * RPQ * SM::ROW_STR);
      __builtin_amdgcn_raw_buffer_store_b128(x, ors, ovoff, i * RPQ * (int)a.so.s * 2, 0);
    }
  };
  if (br.lo > br.hi) {
    // No visible key for any row of this tile: O = 0, LSE = +inf (fwd_kernel.py:327-355)
    if (!first) store_rows(true);
    else if (a.lse && hi == 0 && row_ok) a.lse[lse_offset(si, h, a.hq) + row] = __builtin_inff();
    return;
  }

  // ---- the units (of 32 keys) that these rows see; in the others the two waves only stage and wait
  const int G0 = br.lo, G1 = br.hi;
  int u0 = G0, u1 = G1;
  if (kWindowed) {
    const int64_t cmin = (int64_t)w_rmin - win.left, cmax = (int64_t)w_rmax + win.right;
    if (cmin > 0 && cmin / BN > u0) u0 = (int)(cmin / BN > G1 + 1 ? G1 + 1 : cmin / BN);
    if (cmax < (int64_t)u1 * BN + BN - 1) u1 = cmax < 0 ? -1 : (cmax / BN < u1 ? (int)(cmax / BN) : u1);
  }
  if (wrows <= 0) u1 = G0 - 1;
  u0 = __builtin_amdgcn_readfirstlane(u0);
  u1 = __builtin_amdgcn_readfirstlane(u1);

  // the barrier of a step: what this wave wrote into LDS is there, what it read has arrived
  auto meet = [&]() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };
  auto p_place = [&](int u) { return smem0 + SM::P_OFF + (u & 1) * SM::P_BYTES + w * 2048 + lane * 16; };
  auto factor_place = [&](int u) { return smem0 + SM::FACTOR_OFF + (u & 1) * 1024 + w * 256 + lane * 4; };
  auto keep_place = [&](int u) { return smem0 + SM::KEEP_OFF + (u & 1) * 1024 + w * 256 + lane * 4; };
  const f32x16 zero16 = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};

  constexpr int kRing = 5;      // operands in flight

  // ---- keep bits of the lane's row: four calls per unit, for the columns 8 g + 4 hi .. + 3.  The first wave runs kOwn of them, the second
  // wave the others, of unit u behind its MFMAs in step u
  constexpr int kOwn = 2;
  uint64_t ctr = 0;                              // of the wave's first call of the unit
  uint32_t x_k0 = 0, x_k1 = 0;
  int32_t x_thr = 0;
  Philox px;
  uint32_t word = 0;
  auto keep_begin = [&]() __attribute__((always_inline)) {      // (behind the item's first requests: it waits for the seed)
    if (!kDropout) return;
    const DropoutState ds = make_dropout(a.drop, z, h, a.hq, a.seq.max_seqlen_q, a.seq.max_seqlen_k);
    x_k0 = __builtin_amdgcn_readfirstlane(ds.k0);
    x_k1 = __builtin_amdgcn_readfirstlane(ds.k1);
    x_thr = __builtin_amdgcn_readfirstlane(ds.thr);
    ctr = ds.base + (uint64_t)row * ds.stride + (uint64_t)(G0 * 8 + hi + (first ? 0 : 2 * kOwn));
  };
  auto keep_round = [&](int i, int n) __attribute__((always_inline)) {      // round i % 10 of call i / 10, of n calls
    if (i == 0) word = 0;
    if (i % 10 == 0) {
      const uint64_t at = ctr + (uint64_t)(2 * (i / 10));
      px.start((uint32_t)at, (uint32_t)(at >> 32));
    }
    px.round(i % 10, x_k0, x_k1);
    if (i % 10 == 9) word = dropout_append(px, x_thr, word);
    if (i == 10 * n - 1) ctr += 8;
  };
  if (first) {
    // this lane's Q row, the B operand of S^T = K Q^T
    op_t qreg[KS];
    const T* const q_row = reinterpret_cast<const T*>(a.q) + (int64_t)si.batch_index * a.sq.z + (int64_t)h * a.sq.h +
                           (int64_t)(si.q_start + (row_ok ? row : si.seqlen_q - 1)) * a.sq.s;
    const op_t zero8 = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
    for (int k = 0; k < KS; ++k) qreg[k] = 16 * k + 8 * hi < d_qk ? *reinterpret_cast<const op_t*>(q_row + 16 * k + 8 * hi) : zero8;
    const float qk_scale = a.sm_scale * kLog2e;
    // Fast form: the max is taken on the raw scores and the scale is folded into the exponent, exp2(s*c - m*c), which needs c > 0.
    // With a bias (added after scaling, fwd_kernel_inner.py:166-187) or c <= 0 the scores are scaled first.
    const bool prescale = kBias || !(qk_scale > 0.f);
    const float sc = prescale ? 1.0f : qk_scale;
    float m_i = kNegBig, msc_ref = kNegBig * sc, l_i = 0.f;
    bool have_ref = false;      // every row of the wave has a usable reference maximum

    // ---- bias: 16-byte pieces of the rows, at any alignment, through registers and an area of the wave, requested two units ahead
    // (two sets of registers, and the loads unconditional, so that the wait for one set is not one for the other)
    const bool bias_co = kBias && a.sb_n == 1;
    const T* bias_head = nullptr;
    const T* bias_rows[2];
    op_t bco[2][2];
    if (kBias) {
      bias_head = reinterpret_cast<const T*>(a.bias) + (int64_t)si.batch_index * a.sb_z + (int64_t)h * a.sb_h;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        int m = w_rmin + lane / 4 + 16 * i;
        m = m < si.seqlen_q ? m : si.seqlen_q - 1;
        bias_rows[i] = bias_head + (int64_t)m * a.sb_m + (lane % 4) * 8;
      }
    }
    const int area = smem0 + SM::BIAS_OFF + w * SM::BIAS_BYTES;
    auto bias_fits = [&](int u) { return bias_co && u >= u0 && u <= u1 && (u + 1) * BN <= si.seqlen_k; };
    auto request_bias = [&](auto set, int u) {
      if constexpr (kBias) {
        const bool fits = bias_fits(u);      // (otherwise 16 bytes that are there, for nothing)
#pragma unroll
        for (int i = 0; i < 2; ++i) __builtin_memcpy(&bco[set][i], fits ? bias_rows[i] + u * BN : q_row, 16);
      }
    };
    auto put_bias = [&](auto set) {
      if constexpr (kBias)
#pragma unroll
        for (int i = 0; i < 2; ++i) lds_write(area + set * 4 * SM::BIAS_BYTES + (lane / 4 + 16 * i) * SM::BIAS_ROW + (lane % 4) * 16, bco[set][i]);
    };
    auto bias_read = [&](int set, int q) { return lds_read<q4_t>(area + set * 4 * SM::BIAS_BYTES + c * SM::BIAS_ROW + (8 * q + 4 * hi) * 2); };

    // every key of the unit is visible to every valid row of the wave
    auto sees_all = [&](int u) -> bool {
      const int n_first = u * BN, n_last = u * BN + BN - 1;
      bool all = n_last < si.seqlen_k;
      if (kWindowed) all = all && n_last <= w_rmin + win.right && n_first >= w_rmax - win.left;
      return all;
    };
    // visible columns of this lane's row as one range [m_lo, m_lo + m_rng] (none: m_none)
    int m_lo = 0, m_hi = si.seqlen_k - 1;
    if (kWindowed) {
      m_lo = row - win.left > 0 ? row - win.left : 0;
      m_hi = row + win.right < m_hi ? row + win.right : m_hi;
    }
    const bool m_none = m_hi < m_lo;
    const unsigned m_rng = m_none ? 0u : (unsigned)(m_hi - m_lo);

    int k_at = smem0 + Swz<D>::row_base(lane), k_stage = 0;
    auto k_read = [&](int k) { return lds_read<op_t>((k_at ^ ((k & 7) << 5)) + (k >> 3) * 256); };

    // Two p's, with dropout, in the operand that they become (P is cast to V's dtype for the second GEMM, :274); the operand's eight
    // together go to the second wave
    op_t pb;
    uint32_t keep = 0;
    auto put_pair = [&](int u, int e, float p0, float p1) __attribute__((always_inline)) {
      if (kDropout) {
        int k0, k1;      // the keep bits (the first one uppermost of sixteen) spread over a register
        asm("v_bfe_i32 %0, %1, %2, 1" : "=v"(k0) : "v"(keep), "n"(15 - e));
        asm("v_bfe_i32 %0, %1, %2, 1" : "=v"(k1) : "v"(keep), "n"(14 - e));
        p0 = __builtin_bit_cast(float, __builtin_bit_cast(int, p0) & k0);
        p1 = __builtin_bit_cast(float, __builtin_bit_cast(int, p1) & k1);
      }
      const typename Tr::p2_t p2 = Tr::cvt2(p0, p1);
      pb[e % 8] = p2[0];
      pb[e % 8 + 1] = p2[1];
      if (e % 8 == 6) lds_write(p_place(u) + e / 8 * 1024, pb);
    };
    // Full online-softmax step on the raw scores: scale, bias, mask, row maximum, lazy move of the reference, exponentials, row sum.
    auto softmax_full = [&](int set, int u, f32x16 x) {
      if (prescale) {
#pragma unroll
        for (int i = 0; i < 16; ++i) x[i] *= qk_scale;
      }
      if (kBias) {
        if (bias_fits(u)) {
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const q4_t b4 = bias_read(set, q);
#pragma unroll
            for (int r = 0; r < 4; ++r) x[4 * q + r] += (float)b4[r] * kLog2e;   // fwd_kernel_inner.py:187
          }
        } else {
          const T* bp = bias_head + (int64_t)(row_ok ? row : si.seqlen_q - 1) * a.sb_m;
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            int n = u * BN + 8 * (i / 4) + 4 * hi + (i % 4);
            n = n < si.seqlen_k ? n : si.seqlen_k - 1;
            x[i] += (float)bp[(int64_t)n * a.sb_n] * kLog2e;   // fwd_kernel_inner.py:187
          }
        }
      }
      if (!sees_all(u)) {
        const unsigned d = m_none ? 0x40000000u : (unsigned)(u * BN + 4 * hi - m_lo);
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const bool vis = d + (unsigned)(8 * (i / 4) + (i % 4)) <= m_rng;
          x[i] = vis ? x[i] : -__builtin_inff();
        }
      }
      float mx = x[0];
#pragma unroll
      for (int i = 1; i < 16; ++i) mx = fmaxf(mx, x[i]);
      mx = cross_max(mx);
      // (lazy rescaling, huge scores: see fwd_item)
      const float m_cand = fmaxf(m_i, mx);
      const bool upd = (m_cand - m_i) * sc > 8.0f;
      const float m_new = upd ? m_cand : m_i;
      const float alpha = fast_exp2((m_i - m_new) * sc);
      const float msc = m_new * sc;
      m_i = m_new;
      msc_ref = msc;
      const bool big = __builtin_amdgcn_ballot_w64(!(__builtin_fabsf(msc) < 1024.f)) != 0;
      float rs = 0.f, p[16];
      if (big) {
#pragma unroll
        for (int i = 0; i < 16; ++i) p[i] = fast_exp2((x[i] - m_new) * sc);
      } else {
#pragma unroll
        for (int i = 0; i < 16; ++i) p[i] = fast_exp2(__builtin_fmaf(x[i], sc, -msc));
      }
      // the row sum is over the fp32, undropped p (fwd_kernel_inner.py:213-214)
#pragma unroll
      for (int i = 0; i < 16; ++i) rs += p[i];
      l_i = l_i * alpha + rs;
#pragma unroll
      for (int e = 0; e < 16; e += 2) put_pair(u, e, p[e], p[e + 1]);
      lds_write(factor_place(u), alpha);
      have_ref = !big;
    };

    const bool spec = kBias ? bias_co : !prescale;
    using even = std::integral_constant<int, 0>;
    using odd = std::integral_constant<int, 1>;
    request_bias(even{}, G0);
    request_bias(odd{}, G0 + 1);
    keep_begin();
    __builtin_amdgcn_s_waitcnt(0x0F70);      // (before the steps: the compiler otherwise waits in each of them for Q to have arrived)
    meet();                                  // the first two units of K are there
    f32x16 x = zero16;                       // raw scores of the unit before the running one
    auto step = [&](auto set, int u) __attribute__((always_inline)) {
      const bool act = u >= u0 && u <= u1;
      bool full = u > u0 && u - 1 <= u1;      // there is a unit whose softmax is still to be done in full
      f32x16 acc = zero16;
      op_t ka[kRing];
      if (kDropout) keep = word << (16 - 4 * kOwn) | lds_read<uint32_t>(keep_place(u - 1));      // (of the unit before)
      // behind MFMA k: the unit's bias into its area, the one after the next requested; the first calls of its keep bits
      auto behind = [&](int k) __attribute__((always_inline)) {
        if (k == 8) {
          put_bias(set);
          request_bias(set, u + 2);
        }
        if (kDropout)
#pragma unroll
          for (int i = first_of(k, 10 * kOwn, KS); i < first_of(k + 1, 10 * kOwn, KS); ++i) keep_round(i, kOwn);
        __builtin_amdgcn_sched_barrier(0);
      };
      if (act) {
#pragma unroll
        for (int k = 0; k < kRing - 1; ++k) ka[k] = k_read(k);
      }
      if (act && full && have_ref && spec && sees_all(u - 1)) {
        // Speculative step: the exponentials are taken against the reference the rows have; the row sum tells whether a p left the
        // comfortable range of the 16-bit operand (also inf and NaN), and the unit is then done in full from the raw scores.
        float rs = 0.f, p_even = 0.f;
        q4_t b4[4];
        if (kBias)
#pragma unroll
          for (int q = 0; q < 4; ++q) b4[q] = bias_read(1 - set, q);
#pragma unroll
        for (int k = 0; k < KS; ++k) {
          if (k + kRing - 1 < KS) ka[(k + kRing - 1) % kRing] = k_read(k + kRing - 1);
          acc = Tr::mfma(ka[k % kRing], qreg[k], k == 0 ? zero16 : acc);
          __builtin_amdgcn_sched_barrier(0);
          const float p = fast_exp2(__builtin_fmaf(x[k], qk_scale, kBias ? __builtin_fmaf((float)b4[k / 4][k % 4], kLog2e, -msc_ref) : -msc_ref));
          rs += p;
          if (k % 2 == 0) p_even = p;
          else put_pair(u - 1, k - 1, p_even, p);
          behind(k);
        }
        full = __builtin_amdgcn_ballot_w64(!(rs < 4096.f)) != 0;
        if (!full) {
          l_i += rs;
          lds_write(factor_place(u - 1), 1.0f);
        }
      } else if (act) {
#pragma unroll
        for (int k = 0; k < KS; ++k) {
          if (k + kRing - 1 < KS) ka[(k + kRing - 1) % kRing] = k_read(k + kRing - 1);
          acc = Tr::mfma(ka[k % kRing], qreg[k], k == 0 ? zero16 : acc);
          behind(k);
        }
      } else {
        put_bias(set);
        request_bias(set, u + 2);
        if (kDropout) ctr += 8;
      }
      if (full) softmax_full(1 - set, u - 1, x);
      x = acc;
      k_stage = k_stage == SM::STAGES - 1 ? 0 : k_stage + 1;
      k_at += k_stage == 0 ? (1 - SM::STAGES) * SM::TILE_BYTES : SM::TILE_BYTES;
      meet();
    };
#pragma nounroll
    for (int u = G0; u <= G1 + 1; ++u) {
      step(even{}, u);
      if (kBias) {
        if (++u > G1 + 1) break;
        step(odd{}, u);
      }
    }
    const float l = cross_sum(l_i);
    const bool alive = l > 0.f;
    float inv = alive ? 1.0f / l : 0.f;
    if (kDropout) inv *= 1.0f / (1.0f - a.drop.p);          // fwd_kernel.py:573-575
    lds_write(factor_place(G1 + 1), inv);
    if (a.lse && row_ok && hi == 0)
      a.lse[lse_offset(si, h, a.hq) + row] = alive ? (m_i * sc + fast_log2(l)) * kLn2 : __builtin_inff();   // fwd_kernel.py:610-612
    meet();
    meet();
  } else {
    // ---- staging: K two units ahead of the first waves, V two ahead of this one's use ----------------
    const int tid = threadIdx.x & 255;
    constexpr int LPR = D / 8, RPI = 256 / LPR, RWI = 64 / LPR, CH = BN / RPI;
    static_assert(RPI == 8 && CH == 4, "the swizzle repeats every two accesses");
    const int r0 = tid / LPR, cc0 = tid % LPR;
    int k_voff[2], v_voff[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int gch = cc0 ^ Swz<D>::f(r0 + i * RPI);
      k_voff[i] = gch * 8 < d_qk ? r0 * (int)a.sk.s * 2 + gch * 16 : kVoffOutOfRange;
      v_voff[i] = gch * 8 < d_v ? r0 * (int)a.sv.s * 2 + gch * 16 : kVoffOutOfRange;
    }
    const int k_row = own_scalar((int)a.sk.s * 2), v_row = own_scalar((int)a.sv.s * 2);
    const char* kt = reinterpret_cast<const char*>(a.k) + ((int64_t)si.batch_index * a.sk.z + (int64_t)hk * a.sk.h + (int64_t)(si.k_start + G0 * BN) * a.sk.s) * 2;
    const char* vt = reinterpret_cast<const char*>(a.v) + ((int64_t)si.batch_index * a.sv.z + (int64_t)hk * a.sv.h + (int64_t)(si.k_start + G0 * BN) * a.sv.s) * 2;
    const int rows_all = (si.seqlen_k < (G1 + 1) * BN ? si.seqlen_k : (G1 + 1) * BN) - G0 * BN;
    int k_left = rows_all, v_left = rows_all, k_st = 0, v_st = 0;
    // (a CU takes 16 cycles for each of these loads: they stand between the MFMAs, two at a time)
    u32x4_t k_rs, v_rs;
    auto request_begin = [&](bool both) __attribute__((always_inline)) {
      const int kr = k_left < 0 ? 0 : k_left < BN ? k_left : BN;
      k_rs = wave_rsrc_words(kt, rows_extent(kr, k_row, d_qk * 2));
      if (!both) return;
      const int vr = v_left < 0 ? 0 : v_left < BN ? v_left : BN;
      v_rs = wave_rsrc_words(vt, rows_extent(vr, v_row, d_v * 2));
    };
    auto request_k = [&](int i) __attribute__((always_inline)) {
      const int at = smem0 + k_st * SM::TILE_BYTES + w * RWI * ROWB + i * RPI * ROWB;
      load_to_lds(k_rs, k_voff[0], i * RPI * k_row, at, k_voff[1], (i + 1) * RPI * k_row, at + RPI * ROWB);
    };
    auto request_v = [&](int i) __attribute__((always_inline)) {
      const int at = smem0 + SM::V_OFF + v_st * SM::TILE_BYTES + w * RWI * ROWB + i * RPI * ROWB;
      load_to_lds(v_rs, v_voff[0], i * RPI * v_row, at, v_voff[1], (i + 1) * RPI * v_row, at + RPI * ROWB);
    };
    auto request_end = [&](bool both) __attribute__((always_inline)) {
      kt += (int64_t)BN * k_row;
      k_left -= BN;
      k_st = k_st == SM::STAGES - 1 ? 0 : k_st + 1;
      if (!both) return;
      vt += (int64_t)BN * v_row;
      v_left -= BN;
      v_st = v_st == SM::STAGES - 1 ? 0 : v_st + 1;
    };

    f32x16 o[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int i = 0; i < 16; ++i) o[db][i] = 0.f;

#pragma unroll
    for (int n = 0; n < 2; ++n) {            // units G0, G0 + 1
      request_begin(false);
#pragma unroll
      for (int i = 0; i < CH; i += 2) request_k(i);
      request_end(false);
    }
    keep_begin();
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    meet();
    int v_at = smem0 + SM::V_OFF + Swz<D>::tr_base(lane, 0), v_stage = 0;
    auto v_read = [&](int i) {
      const int t = i / DB, db = i % DB, off = t * 16 * ROWB + (db >> 2) * 256;
      const q4_t x = __builtin_bit_cast(q4_t, lds_read_tr_at((v_at ^ ((db & 3) << 6)) + off));
      const q4_t y = __builtin_bit_cast(q4_t, lds_read_tr_at((v_at ^ ((db & 3) << 6 | 32)) + (off + 8 * ROWB)));
      return __builtin_shufflevector(x, y, 0, 1, 2, 3, 4, 5, 6, 7);
    };
    // step of unit u: O^T += V(u - 2)^T P(u - 2)^T, with the keep bits of unit u behind its MFMAs
    auto end = [&](int u) __attribute__((always_inline)) {
      if (u >= G0 + 2) {
        v_stage = v_stage == SM::STAGES - 1 ? 0 : v_stage + 1;
        v_at += v_stage == 0 ? (1 - SM::STAGES) * SM::TILE_BYTES : SM::TILE_BYTES;
      }
      if (u > G1 + 1) return;
      if (kDropout) lds_write(keep_place(u), word);
      // (this step's requests, eight, are for the step after the next)
      request_end(true);
      asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
      meet();
    };
    auto without_unit = [&](int u) __attribute__((always_inline)) {
      request_begin(true);
#pragma unroll
      for (int i = 0; i < CH; i += 2) { request_k(i); request_v(i); }
      if (kDropout) {
        if (u >= u0 && u <= u1) {
#pragma nounroll
          for (int n = 0; n < 4 - kOwn; ++n) {
            const uint64_t at = ctr + (uint64_t)(2 * n);
            px.start((uint32_t)at, (uint32_t)(at >> 32));
#pragma unroll
            for (int i = 0; i < 10; ++i) px.round(i, x_k0, x_k1);
            word = dropout_append(px, x_thr, n == 0 ? 0u : word);
          }
        }
        ctr += 8;
      }
      end(u);
    };
    int u = G0;
#pragma nounroll
    for (; u < u0 + 2 && u <= G1 + 2; ++u) without_unit(u);
#pragma nounroll
    for (; u <= u1 + 2; ++u) {
      request_begin(true);
      // (units u and u - 2 have their places in common)
      const float f = lds_read<float>(factor_place(u));
      op_t pb[2], va[kRing];
#pragma unroll
      for (int t = 0; t < 2; ++t) pb[t] = lds_read<op_t>(p_place(u) + t * 1024);
#pragma unroll
      for (int i = 0; i < kRing - 1; ++i) va[i] = v_read(i);
      // what O holds so far belongs to the old reference
      if (__builtin_amdgcn_ballot_w64(f != 1.0f) != 0) {
#pragma unroll
        for (int db = 0; db < DB; ++db)
#pragma unroll
          for (int i = 0; i < 16; ++i) o[db][i] *= f;
      }
#pragma unroll
      for (int i = 0; i < 2 * DB; ++i) {
        if (i + kRing - 1 < 2 * DB) va[(i + kRing - 1) % kRing] = v_read(i + kRing - 1);
        o[i % DB] = Tr::mfma(va[i % kRing], pb[i / DB], o[i % DB]);
        if (i % 4 == 1) {
          if (i / 4 < CH / 2) request_k(i / 4 * 2);
          else request_v(i / 4 * 2 - CH);
        }
        if (kDropout)
#pragma unroll
          for (int j = first_of(i, 10 * (4 - kOwn), 2 * DB); j < first_of(i + 1, 10 * (4 - kOwn), 2 * DB); ++j) keep_round(j, 4 - kOwn);
        __builtin_amdgcn_sched_barrier(0);
      }
      end(u);
    }
#pragma nounroll
    for (; u <= G1 + 2; ++u) without_unit(u);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");      // (requests past the last unit, before the rows take their place)
    meet();
    // ---- out: O / l as whole rows, through LDS
    const float inv = lds_read<float>(factor_place(G1 + 1));
    meet();
    const int rows_at = smem0 + w * 32 * SM::ROW_STR + c * SM::ROW_STR + 8 * hi;
#pragma unroll
    for (int db = 0; db < DB; ++db) {
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        q4_t x;
#pragma unroll
        for (int r = 0; r < 4; ++r) x[r] = Tr::cvt(o[db][4 * g + r] * inv);
        lds_write(rows_at + (32 * db + 8 * g) * 2, x);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    store_rows(false);
  }
  __syncthreads();     // the next item reuses LDS
}

}  // namespace fa
