// Forward whose waves own 64 rows instead of 32 (fa_fwd_impl.h): head dims above 64 and up to 128, 16-bit types, no bias, no
// dropout, a positive scale.  Same products, masks and work lists, the same speculative softmax.
//
// The kernel with 32 rows per wave runs two waves per SIMD, which fill each other's gaps, and pays for it with two LDS reads
// per MFMA where one would do.  Here one wave per SIMD works on three units of 32 keys at once: in one stream of instructions
// S of unit g + 1, the exponentials of unit g and PV of unit g - 1, an element behind every MFMA and its three parts
// (exponent, power, sum) behind different ones.  O is accumulated by MFMAs written as asm, Q stays in accumulation registers
// too, scores and P in vector registers (fa_wide.h); three stages of 64-key tiles, one barrier per tile between its units.
// Where a unit needs a new reference maximum its scores are formed again and it takes a full step; the units around it
// are not touched.
//
// Measured (bf16, D128, us, 32-row kernel -> this; one box): B8 H16 S4096 full 968 -> 908, causal 535 -> 522, B1 H32 S16384 causal
// 1930 -> 1830, 1024 queries of 16384 keys Hq 32 Hk 8 262 -> 248.  What bounds it is what the wave issues: per unit 32 MFMAs (512
// cycles of its port), 112 vector instructions (610), 24 LDS reads; 1570 cycles, of which the matrix pipe is busy 65 % (52-54 % of
// the wave time of whole launches, with masked tiles and the ends of items).
// The parts of an element behind one MFMA: 2 % slower; the rows and the first tile of the next item requested before the results
// go out: level (full, 512 keys: 4 % faster; long items 1 % slower).
#pragma once
#include "fa_combine.h"
#include "fa_fwd_impl.h"
#include "fa_wide.h"

namespace fa {

struct WideFwdSmem {
  static constexpr int TILE_BYTES = 64 * 128 * 2;
  static constexpr int STAGE_BYTES = 2 * TILE_BYTES;            // K, V (swizzled)
  static constexpr int Q_OFF = STAGE_BYTES;                     // the item's Q rows on their way to registers; then stages 1 and 2
  static constexpr int AREA_ROW = 256 + 16;
  static constexpr int AREA_OFF = 3 * STAGE_BYTES;              // O rows on their way out, 32 at a time per wave
  static constexpr int BYTES = AREA_OFF + 4 * 32 * AREA_ROW;
  static_assert(Q_OFF + 256 * 256 <= AREA_OFF, "Q fits");
};

// Tile mt (256 rows of head h of sequence z) against all its visible key tiles, with kSplit against part `split` of them: the
// fp32 sums and the row statistics of the part then go to scratch memory, where combine_rows_kernel picks them up.
template <typename T, bool kWindowed, int kPad, bool kSplit>
__device__ __forceinline__ void fwd_wide_item(const FwdArgs& a, const int z, const int h, const int mt, const int split, char* smem_raw) {
  constexpr int D = 128, BM = 256, BN = 64, QB = 2;
  using Tr = Traits<T>;
  using op_t = typename Tr::op_t;
  using q4_t = typename Tr::q4_t;
  using SM = WideFwdSmem;
  constexpr int DC = kPad ? kPad : D;            // columns computed; those past a tensor's head dim are zero
  constexpr int KS = DC / 16, DB = DC / 32, P = KS;      // P: operands (and pairs of MFMAs) of S and of PV per 32 keys
  static_assert(P == 2 * DB, "as many of either");
  constexpr int ROWB = Swz<D>::ROWB;

  const int tid = threadIdx.x;
  const int lane = tid & 63, c = lane & 31, hi = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int d_qk = kPad ? a.head_dim : D, d_v = kPad ? a.head_dim_v : D;

  const SeqInfo si = uniform(get_seq(a.seq, z));
  const int q0 = mt * BM;
  if (q0 >= si.seqlen_q) return;

  Window w{0, 0};
  if (kWindowed) w = parse_window(a.mask.causal_type, a.mask.window_left, a.mask.window_right, si.seqlen_q, si.seqlen_k);
  w.left = w.left > (1 << 30) ? (1 << 30) : (w.left < -(1 << 30) ? -(1 << 30) : w.left);
  w.right = w.right > (1 << 30) ? (1 << 30) : (w.right < -(1 << 30) ? -(1 << 30) : w.right);
  BlockRanges br = block_ranges(kWindowed, w.left, w.right, q0, si.seqlen_q, si.seqlen_k, BM, BN);
  if (kSplit && br.lo <= br.hi) {
    const int per = (br.hi - br.lo + a.splits) / a.splits;
    br.lo += split * per;
    if (br.lo + per - 1 < br.hi) br.hi = br.lo + per - 1;
  }
  const int qw = q0 + 64 * wave;
  const BlockRanges wr = block_ranges(kWindowed, w.left, w.right, qw, si.seqlen_q, si.seqlen_k, 64, BN);

  const int hk = h / (a.hq / a.hk);
  const int row0 = qw + c;                       // this lane's queries: row0 and row0 + 32
  const int row4 = lane / 16, ch = lane % 16;
  const int rows_q = si.seqlen_q - qw < 64 ? si.seqlen_q - qw : 64;      // rows of this wave (<= 0: none)
  float* lse_ptr = a.lse ? a.lse + lse_offset(si, h, a.hq) : nullptr;

  char* area = smem_raw + SM::AREA_OFF + wave * 32 * SM::AREA_ROW;
  T* o_w = reinterpret_cast<T*>(a.out) + (int64_t)si.batch_index * a.so.z + (int64_t)h * a.so.h + (int64_t)(si.q_start + qw) * a.so.s;
  auto store_block = [&](int b) __attribute__((always_inline)) {
    const int rows = rows_q - 32 * b;
    const auto rs = wave_rsrc(o_w + 32 * b * a.so.s, rows > 0 ? ((rows - 1) * (int)a.so.s + d_v) * 2 : 0);
    const int voff = ch * 8 < d_v ? row4 * (int)a.so.s * 2 + ch * 16 : kVoffOutOfRange;
#pragma unroll
    for (int i = 0; i < 8; ++i)
      __builtin_amdgcn_raw_buffer_store_b128(*reinterpret_cast<const u32x4_t*>(area + (row4 + 4 * i) * SM::AREA_ROW + ch * 16), rs,
                                             voff, i * 4 * (int)a.so.s * 2, 2);
  };
  const int64_t part_row = kSplit ? (((int64_t)z * a.hq + h) * a.num_m_tiles + mt) * (int64_t)(a.splits * BM) + split * BM + wave * 64 + c : 0;
  if (br.lo > br.hi) {      // no visible key for any row of this tile: O = 0, LSE = +inf (fwd_kernel.py:327-355)
    if (kSplit) {
#pragma unroll
      for (int b = 0; b < QB; ++b)
        if (row0 + 32 * b < si.seqlen_q && hi == 0) {
          a.part_ml[(part_row + 32 * b) * 2] = kNegBig;
          a.part_ml[(part_row + 32 * b) * 2 + 1] = 0.f;
        }
      return;
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) *reinterpret_cast<u32x4_t*>(area + (row4 + 4 * i) * SM::AREA_ROW + ch * 16) = u32x4_t{0, 0, 0, 0};
#pragma unroll
    for (int b = 0; b < QB; ++b) {
      store_block(b);
      if (lse_ptr && hi == 0 && row0 + 32 * b < si.seqlen_q) lse_ptr[row0 + 32 * b] = __builtin_inff();
    }
    return;
  }

  // ---- staging: K and V tiles of 64 keys in three stages (fa_bwd_wide.h) ------------------------------------------
  const int smem0 = lds_offset(smem_raw);
  const int r0 = tid / 16, gch = ch ^ Swz<D>::f(r0);
  const int k_voff = gch * 8 < d_qk ? r0 * (int)a.sk.s * 2 + gch * 16 : kVoffOutOfRange;
  const int v_voff = gch * 8 < d_v ? r0 * (int)a.sv.s * 2 + gch * 16 : kVoffOutOfRange;
  const int k_row = (int)a.sk.s * 2, v_row = (int)a.sv.s * 2;
  const T* kb = reinterpret_cast<const T*>(a.k) + (int64_t)si.batch_index * a.sk.z + (int64_t)hk * a.sk.h + ((int64_t)si.k_start + (int64_t)br.lo * BN) * a.sk.s;
  const T* vb = reinterpret_cast<const T*>(a.v) + (int64_t)si.batch_index * a.sv.z + (int64_t)hk * a.sv.h + ((int64_t)si.k_start + (int64_t)br.lo * BN) * a.sv.s;
  int f_tiles = br.hi - br.lo + 1, f_rows = si.seqlen_k - br.lo * BN;
  u32x4_t k_rs, v_rs;
  auto fetch_begin = [&]() __attribute__((always_inline)) {
    const int rows = f_tiles > 0 ? min(f_rows, BN) : 0;
    k_rs = wave_rsrc_words(kb, rows_extent(rows, k_row, d_qk * 2));
    v_rs = wave_rsrc_words(vb, rows_extent(rows, v_row, d_v * 2));
    kb += (int64_t)BN * a.sk.s; vb += (int64_t)BN * a.sv.s;
    f_rows -= BN; --f_tiles;
  };
  auto fetch_piece = [&](int stage, int i) __attribute__((always_inline)) {
    const int half = i & 1, lds = smem0 + stage + i / 2 * SM::TILE_BYTES + wave * 4 * ROWB + half * 32 * ROWB;
    if (i < 2) load_to_lds(k_rs, k_voff, half * 32 * k_row, lds, k_voff, half * 32 * k_row + 16 * k_row, lds + 16 * ROWB);
    else load_to_lds(v_rs, v_voff, half * 32 * v_row, lds, v_voff, half * 32 * v_row + 16 * v_row, lds + 16 * ROWB);
  };
  auto fetch_all = [&](int stage) __attribute__((always_inline)) {
    fetch_begin();
#pragma unroll
    for (int i = 0; i < 4; ++i) fetch_piece(stage, i);
  };

  // ---- the item's Q rows: memory -> LDS -> registers ---------------------------------------------------------
  op_t qreg[QB][KS];
  const int row_a = Swz<D>::row_base(lane);
  {
    const T* qp = reinterpret_cast<const T*>(a.q) + (int64_t)si.batch_index * a.sq.z + (int64_t)h * a.sq.h + (int64_t)(si.q_start + qw) * a.sq.s;
    const auto q_rs = wave_rsrc_words(qp, rows_q > 0 ? ((rows_q - 1) * (int)a.sq.s + d_qk) * 2 : 0);
#pragma unroll
    for (int i = 0; i < 16; i += 2)
      rows_to_lds(q_rs, row4 * (int)a.sq.s * 2, 4 * (int)a.sq.s * 2, d_qk, smem0 + SM::Q_OFF + wave * 64 * ROWB, i);
    fetch_all(0);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    const char* Qt = smem_raw + SM::Q_OFF + wave * 64 * ROWB;
#pragma unroll
    for (int b = 0; b < QB; ++b)
#pragma unroll
      for (int k = 0; k < KS; ++k) qreg[b][k] = swz_read_row<T, D>(Qt, row_a, k, b);
#pragma unroll
    for (int b = 0; b < QB; ++b)
#pragma unroll
      for (int k = 0; k < KS; ++k) asm volatile("" : "+a"(qreg[b][k]));
  }
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");      // the first tile is there, Q has left its area

  f32x16 o[QB][DB];
#pragma unroll
  for (int b = 0; b < QB; ++b)
#pragma unroll
    for (int db = 0; db < DB; ++db) acc_zero<T>(o[b][db]);

  int st_cur = 0, st_nxt = SM::STAGE_BYTES, st_fetch = 2 * SM::STAGE_BYTES;
  fetch_all(st_nxt);

  int m_lo[QB];
  unsigned m_rng[QB];
  bool m_none[QB];
#pragma unroll
  for (int b = 0; b < QB; ++b) {
    const int row = row0 + 32 * b;
    int lo = 0, hi_ = si.seqlen_k - 1;
    if (kWindowed) {
      lo = row - w.left > 0 ? row - w.left : 0;
      hi_ = row + w.right < hi_ ? row + w.right : hi_;
    }
    m_none[b] = hi_ < lo;
    m_rng[b] = m_none[b] ? 0u : (unsigned)(hi_ - lo);
    m_lo[b] = lo;
  }

  float m_i[QB] = {kNegBig, kNegBig}, l_i[QB] = {0.f, 0.f}, l_even[QB] = {0.f, 0.f}, msc[QB] = {0.f, 0.f};      // reference maximum (raw scores), partial row sum, maximum * sc
  bool have_ref = false;
  const float sc = a.sm_scale * kLog2e;      // > 0
  const f32x16 zero16 = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};

  // LDS addresses of K rows (tile ra) and of V^T (tile before, see below)
  int ra[KS], tr[2][DB];
  {
    const int tr_a0 = Swz<D>::tr_base(lane, 0), tr_a1 = Swz<D>::tr_base(lane, 1);
#pragma unroll
    for (int k = 0; k < KS; ++k) ra[k] = smem0 + (row_a ^ (k << 5));
#pragma unroll
    for (int db = 0; db < DB; ++db) { tr[0][db] = smem0 + (tr_a0 ^ (db << 6)); tr[1][db] = smem0 + (tr_a1 ^ (db << 6)); }
  }
  auto k_read = [&](int u, int k) __attribute__((always_inline)) { return lds_read<op_t>(ra[k] + u * 32 * ROWB); };
  auto v_read = [&](int u, int i) __attribute__((always_inline)) {
    const int off = SM::TILE_BYTES + (2 * u + i / DB) * 16 * ROWB;
    const q4_t x = __builtin_bit_cast(q4_t, lds_read_tr_at(tr[0][i % DB] + off));
    const q4_t y = __builtin_bit_cast(q4_t, lds_read_tr_at(tr[1][i % DB] + off));
    return __builtin_shufflevector(x, y, 0, 1, 2, 3, 4, 5, 6, 7);
  };
  auto move_k = [&](int step) __attribute__((always_inline)) {
#pragma unroll
    for (int k = 0; k < KS; ++k) { ra[k] += step; asm("" : "+v"(ra[k])); }
  };
  auto move_v = [&](int step) __attribute__((always_inline)) {
#pragma unroll
    for (int db = 0; db < DB; ++db) {
      tr[0][db] += step; asm("" : "+v"(tr[0][db]));
      tr[1][db] += step; asm("" : "+v"(tr[1][db]));
    }
  };

  // Units of 32 keys, two per tile.  A step works on three of them at once: S of unit g + 1, the exponentials of unit g,
  // PV of unit g - 1; unit g of parity U has its scores in s[U] and its P in pb[U].
  f32x16 s[2][QB];
  op_t pb[2][QB][2];
  op_t xk[3], xv[3];
  auto mask_at = [&](int b, int key) __attribute__((always_inline)) -> unsigned { return m_none[b] ? 0x40000000u : (unsigned)(key + 4 * hi - m_lo[b]); };

  // full online-softmax step of unit U at key n0, whose scores are in s[U] (NU = 2: of both units)
  auto full_step = [&](auto first_tag, auto nu_tag, int n0) __attribute__((always_inline)) {
    constexpr int U0 = decltype(first_tag)::value, NU = decltype(nu_tag)::value;
    bool big = false, any = false;
    float alpha[QB];
#pragma unroll
    for (int b = 0; b < QB; ++b) {
      float mx = -__builtin_inff();
#pragma unroll
      for (int u = U0; u < U0 + NU; ++u) {
        const unsigned d = mask_at(b, n0 + 32 * (u - U0));
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const bool vis = d + (unsigned)(8 * (i / 4) + i % 4) <= m_rng[b];
          s[u][b][i] = vis ? s[u][b][i] : -__builtin_inff();
          mx = fmaxf(mx, s[u][b][i]);
        }
      }
      mx = cross_max(mx);
      const float m_cand = fmaxf(m_i[b], mx);
      // (the largest probability so far is then exactly 1 before P is rounded)
      const bool upd = m_cand > m_i[b];
      const float m_new = upd ? m_cand : m_i[b];
      alpha[b] = fast_exp2((m_i[b] - m_new) * sc);
      m_i[b] = m_new;
      msc[b] = m_new * sc;
      big = big || __builtin_amdgcn_ballot_w64(!(__builtin_fabsf(msc[b]) < 1024.f)) != 0;
      any = any || __builtin_amdgcn_ballot_w64(upd) != 0;
    }
    have_ref = !big;
#pragma unroll
    for (int b = 0; b < QB; ++b) {
      float rs = 0.f;
#pragma unroll
      for (int u = U0; u < U0 + NU; ++u) {
        if (big) {      // huge scores: the difference first (fwd_kernel_inner.py:197-205)
#pragma unroll
          for (int i = 0; i < 16; ++i) s[u][b][i] = fast_exp2((s[u][b][i] - m_i[b]) * sc);
        } else {
#pragma unroll
          for (int i = 0; i < 16; ++i) s[u][b][i] = fast_exp2(__builtin_fmaf(s[u][b][i], sc, -msc[b]));
        }
#pragma unroll
        for (int i = 0; i < 16; ++i) rs += s[u][b][i];
#pragma unroll
        for (int t = 0; t < 2; ++t) pb[u][b][t] = pack8<T>(s[u][b], t);
      }
      l_i[b] = l_i[b] * alpha[b] + rs;
    }
    if (NU == 1 && any) {      // (the first step finds sums of zero)
#pragma unroll
      for (int b = 0; b < QB; ++b)
#pragma unroll
        for (int db = 0; db < DB; ++db) acc_scale(o[b][db], alpha[b]);
    }
  };
  // S of the unit at LDS stage `stage`, parity U, into s[U], nothing behind its MFMAs
  auto plain_s = [&](auto u_tag, int stage) __attribute__((always_inline)) {
    constexpr int U = decltype(u_tag)::value;
#pragma unroll
    for (int k = 0; k < KS; ++k) {
      const op_t x = lds_read<op_t>(smem0 + stage + U * 32 * ROWB + (row_a ^ (k << 5)));
#pragma unroll
      for (int b = 0; b < QB; ++b) s[U][b] = Tr::mfma(x, qreg[b][k], k == 0 ? zero16 : s[U][b]);
    }
  };
  using even = std::integral_constant<int, 0>;
  using odd = std::integral_constant<int, 1>;

  // The matrix work of one step: PV of the unit of parity U ^ 1 before, S of the unit of parity U ^ 1 behind, an operand
  // of K after the operand of V^T (which is there first when a tile begins); `work(i)` behind MFMA i of 4 P.
  auto mfmas = [&](auto u_tag, auto work) __attribute__((always_inline)) {
    constexpr int U = decltype(u_tag)::value, N = U ^ 1;
#pragma unroll
    for (int i = 0; i <= P; ++i) {
      if (i < P) {
        if (i + 2 < P) xv[(i + 2) % 3] = v_read(N, i + 2);
#pragma unroll
        for (int b = 0; b < QB; ++b) {
          mfma_acc<T>(o[b][i % DB], xv[i % 3], pb[N][b][i / DB]);
          work(i == 0 ? b : 4 * i - 2 + b);
        }
      }
      if (i > 0) {
        const int k = i - 1;
        if (k + 2 < P) xk[(k + 2) % 3] = k_read(N, k + 2);
#pragma unroll
        for (int b = 0; b < QB; ++b) {
          s[N][b] = Tr::mfma(xk[k % 3], qreg[b][k], k == 0 ? zero16 : s[N][b]);
          work(i == P ? 4 * P - 2 + b : 4 * i + b);
        }
      }
    }
  };
  // step of unit g (parity U, first key n0): speculative exponentials against the reference the rows have; returns whether
  // they stand (fa_fwd_impl.h: sv_fast)
  auto step = [&](auto u_tag, auto masked_tag, int n0) __attribute__((always_inline)) -> bool {
    constexpr int U = decltype(u_tag)::value;
    constexpr bool masked = decltype(masked_tag)::value;
    // (the row sum of a tile is formed over both its units before it meets the row's: the sums of the 32-row kernel, to the bit)
    float rs[QB] = {U == 0 ? 0.f : l_even[0], U == 0 ? 0.f : l_even[1]};
    const unsigned d[QB] = {mask_at(0, n0), mask_at(1, n0)};
    if (U == 1) fetch_begin();
    // an element's three parts stand behind different MFMAs: none waits for the result of the one before
    constexpr int kLag = 2;
    auto exponent = [&](int E) __attribute__((always_inline)) {
      const int b = E / 16, i = E % 16;
      float x = __builtin_fmaf(s[U][b][i], sc, -msc[b]);
      if (masked) {
        const bool vis = d[b] + (unsigned)(8 * (i / 4) + i % 4) <= m_rng[b];
        x = vis ? x : -__builtin_inff();
      }
      s[U][b][i] = x;
    };
    auto power = [&](int E) __attribute__((always_inline)) { s[U][E / 16][E % 16] = fast_exp2(s[U][E / 16][E % 16]); };
    auto sum = [&](int E) __attribute__((always_inline)) {
      const int b = E / 16, i = E % 16;
      rs[b] += s[U][b][i];      // the row sum is over the fp32 p (fwd_kernel_inner.py:213-214)
      if (i & 1) {
        const typename Tr::p2_t p2 = Tr::cvt2(s[U][b][i - 1], s[U][b][i]);
        pb[U][b][i / 8][i % 8 - 1] = p2[0];
        pb[U][b][i / 8][i % 8] = p2[1];
      }
    };
    mfmas(u_tag, [&](int slot) __attribute__((always_inline)) {
      if (U == 1 && slot < 8 && slot % 2 == 1) fetch_piece(st_nxt, slot / 2);
#pragma unroll
      for (int E = first_of(slot, 32 + kLag, 4 * P); E < first_of(slot + 1, 32 + kLag, 4 * P); ++E) {
        if (E < 32) exponent(E);
        if (E >= kLag / 2 && E < 32 + kLag / 2) power(E - kLag / 2);
        if (E >= kLag && E < 32 + kLag) sum(E - kLag);
      }
      __builtin_amdgcn_sched_barrier(0);
    });
    // (complete here; left alone the compiler sinks what the branches below do not need into their targets)
    asm volatile("" : "+v"(rs[0]), "+v"(rs[1]));
#pragma unroll
    for (int b = 0; b < QB; ++b) asm volatile("" : "+v"(pb[U][b][0]), "+v"(pb[U][b][1]));
    // (also catches inf and NaN)
    if (!have_ref || __builtin_amdgcn_ballot_w64(!(rs[0] < 4096.f && rs[1] < 4096.f)) != 0) return false;
#pragma unroll
    for (int b = 0; b < QB; ++b) (U == 0 ? l_even : l_i)[b] = U == 0 ? rs[b] : l_i[b] + rs[b];
    return true;
  };
  // Between the two steps of a tile: the next tile has landed (requested a tile ago) and every wave has left the one before,
  // whose stage is filled again.  K addresses move on; those of V^T stay with the tile.
  auto meet = [&]() __attribute__((always_inline)) {
    asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier\n\ts_nop 1" ::: "memory");
    move_k(st_nxt - st_cur);
    const int t = st_cur;
    st_cur = st_nxt; st_nxt = st_fetch; st_fetch = t;
    xk[0] = k_read(0, 0);
    xk[1] = k_read(0, 1);
  };
  int st_v = 0;
  auto v_to = [&](int stage) __attribute__((always_inline)) {
    move_v(stage - st_v);
    st_v = stage;
    xv[0] = v_read(0, 0);
    xv[1] = v_read(0, 1);
  };
  auto second_unit = [&]() __attribute__((always_inline)) {
    xv[0] = v_read(1, 0);
    xv[1] = v_read(1, 1);
    xk[0] = k_read(1, 0);
    xk[1] = k_read(1, 1);
  };
  using one = std::integral_constant<int, 1>;
  using two = std::integral_constant<int, 2>;
  auto tile = [&](auto masked_tag, int j) __attribute__((always_inline)) {
    const int cur = st_cur;
    l_even[0] = l_even[1] = 0.f;
    const bool ok0 = step(even{}, masked_tag, j * BN);
    v_to(cur);
    if (!ok0) {
      plain_s(even{}, cur);
      full_step(even{}, one{}, j * BN);
    }
    meet();
    const bool ok1 = step(odd{}, masked_tag, j * BN + 32);
    second_unit();
    if (!ok1) {
      l_i[0] += l_even[0];
      l_i[1] += l_even[1];
      plain_s(odd{}, cur);
      full_step(odd{}, one{}, j * BN + 32);
    }
  };

  // the wave's runs of tiles: skipped, the first one (a full step over its 64 keys settles the reference), masked, whole,
  // masked, skipped; all waves take every barrier
  const int lo = max(wr.lo, br.lo), hi_t = min(wr.hi, br.hi);
  const bool none = wr.lo > wr.hi || lo > hi_t;
  const int j_lo = none ? br.hi + 1 : lo, j_end = none ? br.hi + 1 : hi_t + 1;
  const bool full = wr.fb_lo <= wr.fb_hi;
  const int f_lo = full ? min(max(wr.fb_lo, j_lo), j_end) : j_end, f_end = full ? min(max(wr.fb_hi + 1, f_lo), j_end) : j_end;
  auto skip = [&]() __attribute__((always_inline)) {
    meet();
    fetch_all(st_nxt);
  };
  int j = br.lo;
  for (; j < j_lo; ++j) skip();
  if (j < j_end) {
    const int cur = st_cur;
    plain_s(even{}, cur);
    plain_s(odd{}, cur);
    full_step(even{}, two{}, j * BN);
    v_to(cur);
    meet();
    fetch_all(st_nxt);
    mfmas(odd{}, [](int) __attribute__((always_inline)) {});
    second_unit();
    ++j;
    // (left of a window rows see their first keys here: full steps, so that each settles its reference on all of them)
    for (; j < f_lo; ++j) { have_ref = have_ref && !full; tile(std::true_type{}, j); }
    for (; j < f_end; ++j) tile(std::false_type{}, j);
    for (; j < j_end; ++j) tile(std::true_type{}, j);
    asm volatile("s_nop 1");
#pragma unroll
    for (int i = 0; i < P; ++i) {
      if (i + 2 < P) xv[(i + 2) % 3] = v_read(1, i + 2);
#pragma unroll
      for (int b = 0; b < QB; ++b) mfma_acc<T>(o[b][i % DB], xv[i % 3], pb[1][b][i / DB]);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  for (; j <= br.hi; ++j) skip();
  // (requests past the last tile write zeros into stages nobody reads, but before the next item's are filled)
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  acc_settle(o[0], o[1]);
#pragma unroll
  for (int b = 0; b < QB; ++b) {
    const float l = cross_sum(l_i[b]);
    const bool row_ok = row0 + 32 * b < si.seqlen_q;
    if (kSplit) {
      if (row_ok) {
#pragma unroll
        for (int db = 0; db < DB; ++db)
#pragma unroll
          for (int g = 0; g < 4; ++g)
            *reinterpret_cast<f32x4*>(a.part_o + (part_row + 32 * b) * D + 32 * db + 8 * g + 4 * hi) =
                f32x4{o[b][db][4 * g], o[b][db][4 * g + 1], o[b][db][4 * g + 2], o[b][db][4 * g + 3]};
        if (hi == 0) {
          a.part_ml[(part_row + 32 * b) * 2] = m_i[b];
          a.part_ml[(part_row + 32 * b) * 2 + 1] = l;
        }
      }
      continue;
    }
    const bool alive = l > 0.f;
    const float inv = alive ? 1.0f / l : 0.f;
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        q4_t t4;
#pragma unroll
        for (int r = 0; r < 4; ++r) t4[r] = Tr::cvt(o[b][db][4 * g + r] * inv);
        *reinterpret_cast<q4_t*>(area + c * SM::AREA_ROW + (32 * db + 8 * g + 4 * hi) * 2) = t4;
      }
    __builtin_amdgcn_sched_barrier(0);
    store_block(b);
    __builtin_amdgcn_sched_barrier(0);
    if (row_ok && lse_ptr && hi == 0)
      lse_ptr[row0 + 32 * b] = alive ? (m_i[b] * sc + fast_log2(l)) * kLn2 : __builtin_inff();   // fwd_kernel.py:610-612
  }
}

template <typename T, bool kWindowed, int kPad, bool kSplit>
__global__ __attribute__((amdgpu_flat_work_group_size(256, 256))) __attribute__((amdgpu_waves_per_eu(1, 1)))
void fwd_wide_kernel(const FwdArgs a) {
  extern __shared__ __attribute__((aligned(16))) char smem_raw[];
  const int xcd = blockIdx.x % kNumXcd, p = blockIdx.x / kNumXcd, workers = gridDim.x / kNumXcd;
  const int per_group = a.zh_group * a.num_m_tiles;
  const int ratio = a.hq / a.hk, nseq = a.num_zh / a.hq;
  const bool ragged = a.seq.num_seqlens != 0 && a.zh_per_xcd <= kLevelCap && a.num_m_tiles <= 0xffff;
  const int zh_lo = xcd * a.zh_per_xcd;
  LevelWalk walk;
  if (ragged)
    walk.init<256>(reinterpret_cast<uint32_t*>(smem_raw + WideFwdSmem::BYTES), a.seq, zh_lo,
                   zh_lo + a.zh_per_xcd < a.num_zh ? zh_lo + a.zh_per_xcd : a.num_zh, nseq, ratio, 256, false, threadIdx.x);
  for (int r = 0; r * workers < a.items_per_xcd; ++r) {
    const int t = worker_pos<false>(r, p, workers, a.num_cu);
    int zh, mt, split = 0;
    if (ragged) {
      int e;
      if (!walk.at(t, e, mt)) break;
      zh = zh_lo + e;
    } else {
      if (t >= a.items_per_xcd) continue;
      const int ti = kSplit ? t / a.splits : t;
      split = kSplit ? t % a.splits : 0;
      const int gi = ti / per_group, gr = ti % per_group;
      const int zl = gi * a.zh_group + gr % a.zh_group;
      zh = zh_lo + zl;
      if (zl >= a.zh_per_xcd || zh >= a.num_zh) continue;
      mt = a.num_m_tiles - 1 - gr / a.zh_group;
    }
    int z, h;
    split_zh(zh, nseq, ratio, z, h);
    fwd_wide_item<T, kWindowed, kPad, kSplit>(a, z, h, mt, split, smem_raw);
    __syncthreads();
  }
}

template <typename T, bool W, int kPad, bool kSplit>
hipError_t launch_fwd_wide(const FwdArgs& a, dim3 grid, hipStream_t stream) {
  auto kern = fwd_wide_kernel<T, W, kPad, kSplit>;
  constexpr int smem = WideFwdSmem::BYTES + kLevelBytes;
  static std::atomic<uint64_t> lds_set{0};
  hipError_t e = allow_large_lds(reinterpret_cast<const void*>(kern), smem, lds_set);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(kern, grid, dim3(256), smem, stream, a);
  e = hipGetLastError();
  if (kSplit && e == hipSuccess) e = launch_combine_rows<T, 128>(a, a.num_zh, stream);
  return e;
}

template <typename T, int kPad>
hipError_t launch_fwd_wide_any(const FwdArgs& a, bool windowed, hipStream_t stream) {
  const int nseq = a.seq.num_seqlens != 0 ? (a.seq.num_seqlens < 0 ? -a.seq.num_seqlens : a.seq.num_seqlens) : a.batch;
  FwdArgs b = a;
  b.num_m_tiles = (a.seq.max_seqlen_q + 255) / 256;
  const bool split = a.splits > 1;
  const TileWork w = tile_work(nseq * a.hq, q_head_group(a.hq, a.hk), b.num_m_tiles * (split ? a.splits : 1));
  b.num_zh = w.num_zh; b.zh_per_xcd = w.zh_per_xcd; b.zh_group = w.zh_group; b.items_per_xcd = w.items_per_xcd;
  const dim3 grid((unsigned)(kNumXcd * tile_workers(w.items_per_xcd, a.num_cu, 1)));
  if (grid.x == 0) return hipSuccess;
  if (split) {
    b.part_group = 1; b.part_block = 256; b.part_rows = 256; b.row_blocks = b.num_m_tiles;
    return windowed ? launch_fwd_wide<T, true, kPad, true>(b, grid, stream) : launch_fwd_wide<T, false, kPad, true>(b, grid, stream);
  }
  return windowed ? launch_fwd_wide<T, true, kPad, false>(b, grid, stream) : launch_fwd_wide<T, false, kPad, false>(b, grid, stream);
}

}  // namespace fa
