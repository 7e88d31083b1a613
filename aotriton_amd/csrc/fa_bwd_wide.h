// Backward kernels whose waves own 64 rows instead of 32 (fa_bwd_impl.h): head dims above 64 and up to 128, 16-bit types, no
// bias, no dropout.  Same products, masks and work lists; both recompute S and dP.
//
// What bounds the 32-row kernels is not the matrix pipe but what one wave per SIMD issues next to it, and every operand read
// from LDS serves one MFMA only.  With 64 rows it serves two: half the LDS reads and half the Q/dO (K/V) traffic per FLOP.
// A step is 32 rows of the other side, 64 (dK/dV) or 48 (dQ) MFMAs per wave as before.  The registers for it:
//  * the results (256 / 128 registers) are accumulated by MFMAs written as asm, in accumulation registers; S and dP come from
//    the compiler's own MFMAs in vector registers (-amdgpu-mfma-vgpr-form), where the vector ALU works on them in place.  The
//    32-row dK/dV kernel copies all of S and dP over (64 of its 212 vector instructions per tile);
//  * LDS addresses are carried from stage to stage instead of being formed from a base.
// Around the tile loop: three stages, so that the one barrier of a tile stands in its middle, the first operands of the next
// tile are requested before its end and a fetch has a whole tile to land; fetches are asm as well, because the compiler makes
// the first transposing LDS read behind its own wait for them; the item's rows come in and its results go out as whole rows
// through LDS (an item of the 32-row kernels spends 9 us on that and its other ends, one of these 6).
//
// Measured (bf16, D128, us, 32-row kernel -> this; one box): dK/dV B4 H32 S4096 causal 1125 -> 1000, full 1956 -> 1740, B1 H32
// S16384 causal 3840 -> 3380; dQ 840 -> 735, 1435 -> 1280, 2770 -> 2495.  The clock falls with the load: at length the matrix
// pipe is busy for 63 % / 68 % of the time (53 % / 56 % before) at 1.77 / 1.69 GHz (1.90 / 1.89 before), 1250 / 1290 TFLOP/s; a
// few launches of B4 H32 S4096 causal 57 % / 59 % at about 1.85.  A bf16 product of the library reaches 1220-1270 on this card.  Spreading the vector work differently over the MFMAs is level.
#pragma once
#include "fa_bwd_impl.h"
#include "fa_wide.h"

namespace fa {

constexpr int kWideBM = 32, kWideBN = 256;


struct WideDkDvSmem {
  static constexpr int TILE_BYTES = kWideBM * 128 * 2;
  static constexpr int STAGE_BYTES = 2 * TILE_BYTES + 2 * kWideBM * 4;      // Q, dO (swizzled); -L log2e, -delta
  static constexpr int K_OFF = STAGE_BYTES;            // the item's K rows on their way to registers; then stages 1 and 2
  static constexpr int V_OFF = K_OFF + kWideBN * 256;  // its V rows; at the end dK and dV on their way out
  static constexpr int BYTES = V_OFF + kWideBN * 256;
  static_assert(3 * STAGE_BYTES <= V_OFF, "three stages");
};

template <typename T, bool kWindowed, int kPad>
__device__ __forceinline__ void dkdv_wide_item(const BwdArgs& a, const int hk, const int nt, const int z, char* smem_raw) {
  constexpr int D = 128, BM = kWideBM, BN = kWideBN, KB = 2;
  using Tr = Traits<T>;
  using op_t = typename Tr::op_t;
  using q4_t = typename Tr::q4_t;
  using SM = WideDkDvSmem;
  constexpr int DC = kPad ? kPad : D;            // columns computed; those past a tensor's head dim are zero
  constexpr int KS = DC / 16, DB = DC / 32, TS = BM / 16;
  constexpr int ROWB = Swz<D>::ROWB;

  const int tid = threadIdx.x;
  const int lane = tid & 63, c = lane & 31, hi = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int d_qk = kPad ? a.head_dim : D, d_v = kPad ? a.head_dim_v : D;

  const SeqInfo si = uniform(get_seq(a.seq, z));
  const int n0 = nt * BN;
  if (n0 >= si.seqlen_k) return;

  Window w{0, 0};
  if (kWindowed) w = parse_window(a.mask.causal_type, a.mask.window_left, a.mask.window_right, si.seqlen_q, si.seqlen_k);
  w.left = w.left > (1 << 30) ? (1 << 30) : (w.left < -(1 << 30) ? -(1 << 30) : w.left);
  w.right = w.right > (1 << 30) ? (1 << 30) : (w.right < -(1 << 30) ? -(1 << 30) : w.right);
  const BlockRanges br = block_ranges(kWindowed, w.right, w.left, n0, si.seqlen_k, si.seqlen_q, BN, BM);
  // the query tiles that see keys of this wave (the others it only waits through)
  const int nw = n0 + 64 * wave;
  const BlockRanges wr = block_ranges(kWindowed, w.right, w.left, nw, si.seqlen_k, si.seqlen_q, 64, BM);

  const int group = a.hq / a.hk;
  const int key0 = nw + c;                       // this lane's keys: key0 and key0 + 32
  // lanes of a row access: 16 lanes per row of 256 bytes, 4 rows per wave instruction
  const int row4 = lane / 16, ch = lane % 16;
  const int rows_k = si.seqlen_k - nw < 64 ? si.seqlen_k - nw : 64;      // keys of this wave (<= 0: none)

  // results: 32 rows at a time through LDS, whole rows to memory
  char* area = smem_raw + SM::V_OFF + wave * 64 * ROWB;
  constexpr int AREA_ROW = 256 + 16;
  const int64_t dk0 = (int64_t)si.batch_index * a.sdk.z + (int64_t)hk * a.sdk.h + (int64_t)(si.k_start + nw) * a.sdk.s;
  const int64_t dv0 = (int64_t)si.batch_index * a.sdv.z + (int64_t)hk * a.sdv.h + (int64_t)(si.k_start + nw) * a.sdv.s;
  auto store_block = [&](T* base, int64_t stride, int d, int b) __attribute__((always_inline)) {
    const int rows = rows_k - 32 * b;
    const auto rs = wave_rsrc(base + 32 * b * stride, rows > 0 ? ((rows - 1) * (int)stride + d) * 2 : 0);
    const int voff = ch * 8 < d ? row4 * (int)stride * 2 + ch * 16 : kVoffOutOfRange;
#pragma unroll
    for (int i = 0; i < 8; ++i)
      __builtin_amdgcn_raw_buffer_store_b128(*reinterpret_cast<const u32x4_t*>(area + (row4 + 4 * i) * AREA_ROW + ch * 16), rs,
                                             voff, i * 4 * (int)stride * 2, 0);
  };
  if (br.lo > br.hi) {      // no query sees these keys
#pragma unroll
    for (int i = 0; i < 8; ++i) *reinterpret_cast<u32x4_t*>(area + (row4 + 4 * i) * AREA_ROW + ch * 16) = u32x4_t{0, 0, 0, 0};
#pragma unroll
    for (int b = 0; b < KB; ++b) {
      store_block(reinterpret_cast<T*>(a.dk) + dk0, a.sdk.s, d_qk, b);
      store_block(reinterpret_cast<T*>(a.dv) + dv0, a.sdv.s, d_v, b);
    }
    return;
  }

  int q_lo[KB];
  unsigned q_rng[KB];
  bool q_none[KB];
#pragma unroll
  for (int b = 0; b < KB; ++b) {
    const int key = key0 + 32 * b;
    int lo = 0, hi_ = si.seqlen_q - 1;
    if (kWindowed) {
      lo = key - w.right > 0 ? key - w.right : 0;
      hi_ = key + w.left < hi_ ? key + w.left : hi_;
    }
    q_none[b] = key >= si.seqlen_k || hi_ < lo;
    q_rng[b] = q_none[b] ? 0u : (unsigned)(hi_ - lo);
    q_lo[b] = lo;
  }

  // ---- staging ----------------------------------------------------------------------------
  // Tiles of 32 queries.  (From the last one down, which would let the items of a head that run side by side under a causal
  // mask read the same tiles at the same time, 0-1 % faster; up, sums and results are those of the 128-row kernel.)  Three stages: while a tile is worked on, the next one lands and the one after it is requested
  // (behind the barrier in the middle of the tile, where every wave has left the tile before).
  const int smem0 = lds_offset(smem_raw);
  const int r0 = tid / 16, gch = ch ^ Swz<D>::f(r0);      // row of a tile and 16-byte chunk this lane fetches; rows r0 + 16 too
  const int q_voff = gch * 8 < d_qk ? r0 * (int)a.sq.s * 2 + gch * 16 : kVoffOutOfRange;
  const int do_voff = gch * 8 < d_v ? r0 * (int)a.sdo.s * 2 + gch * 16 : kVoffOutOfRange;
  const int q_row = (int)a.sq.s * 2, do_row = (int)a.sdo.s * 2;
  const int ntq = br.hi - br.lo + 1;
  const T* qb = nullptr; const T* dob = nullptr;
  const float* st_b = nullptr;      // lower half of the lanes: L of the head, upper half: delta
  int f_g = 0, f_e = 0, f_m = 0;      // q-head of the group, tiles left of it (0: nothing left to fetch), first query
  float st_val = 0.f;
  auto set_head = [&]() __attribute__((always_inline)) {
    const int hq = hk * group + f_g;
    const int64_t row0 = (int64_t)si.q_start + (int64_t)br.lo * BM;
    qb = reinterpret_cast<const T*>(a.q) + (int64_t)si.batch_index * a.sq.z + (int64_t)hq * a.sq.h + row0 * a.sq.s;
    dob = reinterpret_cast<const T*>(a.dout) + (int64_t)si.batch_index * a.sdo.z + (int64_t)hq * a.sdo.h + row0 * a.sdo.s;
    st_b = (hi ? a.delta : a.lse) + lse_offset(si, hq, a.hq);
    f_e = ntq;
    f_m = br.lo * BM;
  };
  u32x4_t q_rs, do_rs;
  auto fetch_begin = [&]() __attribute__((always_inline)) {
    // (arithmetic instead of choices, for which the compiler makes branches)
    const int rows = min(f_e > 0 ? si.seqlen_q - f_m : 0, BM);
    q_rs = wave_rsrc_words(qb, rows_extent(rows, q_row, d_qk * 2));
    do_rs = wave_rsrc_words(dob, rows_extent(rows, do_row, d_v * 2));
    // (every wave reads and stores the row statistics: a branch for one of them would split the tile's code into blocks,
    // between which the compiler moves the work that is placed behind the MFMAs)
    st_val = st_b[min(f_m + c, si.seqlen_q - 1)];
  };
  auto fetch_piece = [&](int stage, int i) __attribute__((always_inline)) {
    const int lds = smem0 + stage + i * SM::TILE_BYTES + wave * 4 * ROWB;
    if (i == 0) load_to_lds(q_rs, q_voff, 0, lds, q_voff, 16 * q_row, lds + 16 * ROWB);
    else load_to_lds(do_rs, do_voff, 0, lds, do_voff, 16 * do_row, lds + 16 * ROWB);
  };
  auto fetch_end = [&]() __attribute__((always_inline)) {
    qb += (int64_t)BM * a.sq.s; dob += (int64_t)BM * a.sdo.s;
    f_m += BM;
    if (--f_e == 0 && ++f_g < group) set_head();
  };
  auto fetch_all = [&](int stage) __attribute__((always_inline)) {
    fetch_begin();
#pragma unroll
    for (int i = 0; i < 2; ++i) fetch_piece(stage, i);
    fetch_end();
  };
  const float st_mul = hi ? -1.0f : -kRcpLn2;
  auto store_stats = [&](int stage) __attribute__((always_inline)) {
    *reinterpret_cast<__attribute__((address_space(3))) float*>(smem0 + stage + 2 * SM::TILE_BYTES + lane * 4) = st_val * st_mul;
  };

  // ---- the item's K and V rows: memory -> LDS -> registers
  {
    const T* kb = reinterpret_cast<const T*>(a.k) + (int64_t)si.batch_index * a.sk.z + (int64_t)hk * a.sk.h + (int64_t)(si.k_start + nw) * a.sk.s;
    const T* vb = reinterpret_cast<const T*>(a.v) + (int64_t)si.batch_index * a.sv.z + (int64_t)hk * a.sv.h + (int64_t)(si.k_start + nw) * a.sv.s;
    const auto k_rs = wave_rsrc_words(kb, rows_k > 0 ? ((rows_k - 1) * (int)a.sk.s + d_qk) * 2 : 0);
    const auto v_rs = wave_rsrc_words(vb, rows_k > 0 ? ((rows_k - 1) * (int)a.sv.s + d_v) * 2 : 0);
#pragma unroll
    for (int i = 0; i < 16; i += 2) {
      rows_to_lds(k_rs, row4 * (int)a.sk.s * 2, 4 * (int)a.sk.s * 2, d_qk, smem0 + SM::K_OFF + wave * 64 * ROWB, i);
      rows_to_lds(v_rs, row4 * (int)a.sv.s * 2, 4 * (int)a.sv.s * 2, d_v, smem0 + SM::V_OFF + wave * 64 * ROWB, i);
    }
  }
  set_head();
  fetch_all(0);
  store_stats(0);
  const int row_a = Swz<D>::row_base(lane), tr_a0 = Swz<D>::tr_base(lane, 0), tr_a1 = Swz<D>::tr_base(lane, 1);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  op_t kreg[KB][KS], vreg[KS];      // (V of the second key block stays in LDS: there is no room for it next to the rest)
  const char* Kt = smem_raw + SM::K_OFF + wave * 64 * ROWB;
  const char* Vt = smem_raw + SM::V_OFF + wave * 64 * ROWB;
#pragma unroll
  for (int b = 0; b < KB; ++b)
#pragma unroll
    for (int k = 0; k < KS; ++k) {
      kreg[b][k] = swz_read_row<T, D>(Kt, row_a, k, b);
      if (b == 0) vreg[k] = swz_read_row<T, D>(Vt, row_a, k, b);
    }
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");      // tile 0 is there, K has left its area

  f32x16 dk[KB][DB], dv[KB][DB];
#pragma unroll
  for (int b = 0; b < KB; ++b)
#pragma unroll
    for (int db = 0; db < DB; ++db)
      { acc_zero<T>(dk[b][db]); acc_zero<T>(dv[b][db]); }

  int st_cur = 0, st_nxt = SM::STAGE_BYTES, st_fetch = 2 * SM::STAGE_BYTES;
  fetch_all(st_nxt);

  const float qk_scale = a.sm_scale * kLog2e;
  const f32x16 zero16 = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};

  // LDS addresses of the running tile's operands, moved on from stage to stage (kept as they are: base and offset apart
  // would take twice the registers)
  int ra[KS], tr[2][DB], sa = smem0 + 2 * SM::TILE_BYTES + 16 * hi;
#pragma unroll
  for (int k = 0; k < KS; ++k) ra[k] = smem0 + (row_a ^ (k << 5));
#pragma unroll
  for (int db = 0; db < DB; ++db) { tr[0][db] = smem0 + (tr_a0 ^ (db << 6)); tr[1][db] = smem0 + (tr_a1 ^ (db << 6)); }
  auto rotate = [&]() __attribute__((always_inline)) {
    const int step = st_nxt - st_cur, t = st_cur;
#pragma unroll
    for (int k = 0; k < KS; ++k) { ra[k] += step; asm("" : "+v"(ra[k])); }
#pragma unroll
    for (int db = 0; db < DB; ++db) {
      tr[0][db] += step; asm("" : "+v"(tr[0][db]));
      tr[1][db] += step; asm("" : "+v"(tr[1][db]));
    }
    sa += step; asm("" : "+v"(sa));
    st_cur = st_nxt; st_nxt = st_fetch; st_fetch = t;
  };
  auto q_read = [&](int k) __attribute__((always_inline)) { return lds_read<op_t>(ra[k]); };
  auto do_read = [&](int k) __attribute__((always_inline)) { return lds_read<op_t>(ra[k] + SM::TILE_BYTES); };
  // first operands of a tile, requested at the end of the tile before
  op_t xa[3];
  auto prefetch = [&]() __attribute__((always_inline)) { xa[0] = q_read(0); xa[1] = q_read(1); };
  prefetch();

  auto compute = [&](auto masked_tag, int e) __attribute__((always_inline)) {
    constexpr bool masked = decltype(masked_tag)::value;
    const int m0 = (br.lo + e) * BM;
    auto l_read = [&](int q) __attribute__((always_inline)) { return lds_read<f32x4>(sa + 32 * q); };
    auto d_read = [&](int q) __attribute__((always_inline)) { return lds_read<f32x4>(sa + BM * 4 + 32 * q); };

    f32x16 s[KB], dp[KB], nd = zero16;
    op_t pb[KB][TS], sb[KB][TS];
    f32x4 l4[2];

    // ---- S = Q K^T
    store_stats(st_nxt);
#pragma unroll
    for (int k = 0; k < KS; ++k) {
      xa[(k + 2) % 3] = k + 2 < KS ? q_read(k + 2) : do_read(k + 2 - KS);
      if (k < 4) {
        const f32x4 t4 = d_read(k);
#pragma unroll
        for (int r = 0; r < 4; ++r) nd[4 * k + r] = t4[r];
      }
#pragma unroll
      for (int b = 0; b < KB; ++b) {
        s[b] = Tr::mfma(xa[k % 3], kreg[b][k], k == 0 ? zero16 : s[b]);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    l4[0] = l_read(0);

    unsigned q_d[KB];
#pragma unroll
    for (int b = 0; b < KB; ++b) q_d[b] = q_none[b] ? 0x40000000u : (unsigned)(m0 + 4 * hi - q_lo[b]);
    // elements in the order rows 4 q .. 4 q + 3 of key block 0, then of block 1 (the statistics serve both)
    auto exponent = [&](int E) __attribute__((always_inline)) {
      const int q = E / 8, b = (E / 4) % 2, r = E % 4, i = 4 * q + r;
      if (E % 8 == 0 && q < 3) l4[(q + 1) & 1] = l_read(q + 1);
      float x = __builtin_fmaf(s[b][i], qk_scale, l4[q & 1][r]);
      if (masked) {
        const bool vis = q_d[b] + (unsigned)(8 * q + r) <= q_rng[b];
        x = vis ? x : -__builtin_inff();
      }
      s[b][i] = x;
    };
    auto power = [&](int E) __attribute__((always_inline)) {
      const int b = (E / 4) % 2, i = 4 * (E / 8) + E % 4;
      s[b][i] = fast_exp2(s[b][i]);
    };
    auto p_pair = [&](int E) __attribute__((always_inline)) {      // E odd
      const int q = E / 8, b = (E / 4) % 2, r = E % 4, i = 4 * q + r;
      const typename Tr::p2_t p2 = Tr::cvt2(s[b][i - 1], s[b][i]);
      pb[b][i / 8][i % 8 - 1] = p2[0];
      pb[b][i / 8][i % 8] = p2[1];
    };
    auto ds_el = [&](int E) __attribute__((always_inline)) {
      const int b = (E / 4) % 2, i = 4 * (E / 8) + E % 4;
      dp[b][i] = s[b][i] * dp[b][i];      // (dP started at -delta)
    };
    auto ds_pair = [&](int E) __attribute__((always_inline)) {      // E odd
      const int b = (E / 4) % 2, i = 4 * (E / 8) + E % 4;
      const typename Tr::p2_t s2 = Tr::cvt2(dp[b][i - 1], dp[b][i]);
      sb[b][i / 8][i % 8 - 1] = s2[0];
      sb[b][i / 8][i % 8] = s2[1];
    };
    // one ring of transposed operands runs through dV and dK
    constexpr int G3 = TS * DB, kRing = 4;
    op_t ta[kRing];
    auto ta_read = [&](int i) __attribute__((always_inline)) {
      const int j = i % G3, off = (i < G3 ? SM::TILE_BYTES : 0) + j / DB * 16 * ROWB;
      const q4_t x = __builtin_bit_cast(q4_t, lds_read_tr_at(tr[0][j % DB] + off));
      const q4_t y = __builtin_bit_cast(q4_t, lds_read_tr_at(tr[1][j % DB] + off));
      return __builtin_shufflevector(x, y, 0, 1, 2, 3, 4, 5, 6, 7);
    };

    // ---- dP = dO V^T, with p behind its MFMAs
    op_t vl[2];
    vl[0] = swz_read_row<T, D>(Vt, row_a, 0, 1);
#pragma unroll
    for (int k = 0; k < KS; ++k) {
      if (k + 2 < KS) xa[(KS + k + 2) % 3] = do_read(k + 2);
      if (k + 1 < KS) vl[(k + 1) % 2] = swz_read_row<T, D>(Vt, row_a, k + 1, 1);
      if (k == KS - 1) {
#pragma unroll
        for (int i = 0; i < kRing - 1; ++i) ta[i] = ta_read(i);
      }
#pragma unroll
      for (int b = 0; b < KB; ++b) {
        dp[b] = Tr::mfma(xa[(KS + k) % 3], b == 0 ? vreg[k] : vl[k % 2], k == 0 ? nd : dp[b]);
        const int gi = k * KB + b;
        // (the three parts of an element one after the other behind different MFMAs: none waits for the one before)
        const int E0 = first_of(gi, 34, KS * KB), E1 = first_of(gi + 1, 34, KS * KB);
#pragma unroll
        for (int E = E0; E < E1; ++E) {
          if (E < 32) exponent(E);
          if (E >= 1 && E <= 32) power(E - 1);
          if (E >= 2 && (E & 1)) p_pair(E - 2);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
#pragma unroll
    for (int b = 0; b < KB; ++b)
#pragma unroll
      for (int t = 0; t < TS; ++t) asm volatile("" : "+v"(pb[b][t]));      // (complete here, not sunk to where they are used)
    // the next tile has landed (requested a tile ago), and every wave has left the tile before this one
    asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier\n\ts_nop 1" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);

    // ---- dV^T += dO^T P, with dS and the fetch of the tile after the next behind its MFMAs
#pragma unroll
    for (int i = 0; i < G3; ++i) {
      ta[(i + kRing - 1) % kRing] = ta_read(i + kRing - 1);
#pragma unroll
      for (int b = 0; b < KB; ++b) {
        mfma_acc<T>(dv[b][i % DB], ta[i % kRing], pb[b][i / DB]);
        const int gi = i * KB + b;
        if (gi == 0) fetch_begin();
        if (gi == 1 || gi == 3) fetch_piece(st_fetch, gi / 2);
#pragma unroll
        for (int E = first_of(gi, 34, G3 * KB); E < first_of(gi + 1, 34, G3 * KB); ++E) {
          if (E < 32) ds_el(E);
          if (E >= 2 && (E & 1)) ds_pair(E - 2);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    // ---- dK^T += Q^T dS
    asm volatile("s_nop 1");
#pragma unroll
    for (int i = G3; i < 2 * G3; ++i) {
      if (i + kRing - 1 < 2 * G3) ta[(i + kRing - 1) % kRing] = ta_read(i + kRing - 1);
      if (i == 2 * G3 - kRing + 1) rotate();      // (the last transposed operands are on their way)
      if (i == 2 * G3 - 2) prefetch();
#pragma unroll
      for (int b = 0; b < KB; ++b) mfma_acc<T>(dk[b][i % DB], ta[i % kRing], sb[b][(i - G3) / DB]);
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  // the wave's runs of query tiles, counted from br.lo: skipped, masked, whole, masked, skipped.  Every run has its own loop
  // (a branch around the MFMAs would make the compiler carry the accumulators across it); all waves take every barrier.
  const bool none = wr.lo > wr.hi, full = !none && wr.fb_lo <= wr.fb_hi;
  const int e_lo = none ? ntq : wr.lo - br.lo;
  const int e_end = none ? ntq : wr.hi + 1 - br.lo;
  const int f_lo = full ? wr.fb_lo - br.lo : e_end;
  const int f_end = full ? wr.fb_hi + 1 - br.lo : e_end;
  auto skip = [&]() __attribute__((always_inline)) {
    store_stats(st_nxt);
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    fetch_all(st_fetch);
    rotate();
    prefetch();
  };
  for (int g = 0; g < group; ++g) {
    int e = 0;
    for (; e < e_lo; ++e) skip();
    for (; e < f_lo; ++e) { compute(std::true_type{}, e); fetch_end(); }
    for (; e < f_end; ++e) { compute(std::false_type{}, e); fetch_end(); }
    for (; e < e_end; ++e) { compute(std::true_type{}, e); fetch_end(); }
    for (; e < ntq; ++e) skip();
  }
  // (fetches past the last tile write zeros into stages nobody reads, but before the next item's stages are filled)
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
  for (int b = 0; b < KB; ++b) {
    acc_settle(dk[b], dv[b]);
#pragma unroll
    for (int which = 0; which < 2; ++which) {
#pragma unroll
      for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          q4_t x;
#pragma unroll
          for (int r = 0; r < 4; ++r) x[r] = Tr::cvt(which ? dv[b][db][4 * g + r] : dk[b][db][4 * g + r] * a.sm_scale);
          *reinterpret_cast<q4_t*>(area + c * AREA_ROW + (32 * db + 8 * g + 4 * hi) * 2) = x;
        }
      __builtin_amdgcn_sched_barrier(0);
      if (which) store_block(reinterpret_cast<T*>(a.dv) + dv0, a.sdv.s, d_v, b);
      else store_block(reinterpret_cast<T*>(a.dk) + dk0, a.sdk.s, d_qk, b);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
}

template <typename T, bool kWindowed, int kPad>
__global__ __attribute__((amdgpu_flat_work_group_size(256, 256))) __attribute__((amdgpu_waves_per_eu(1, 1)))
void bwd_dkdv_wide_kernel(const BwdArgs a) {
  extern __shared__ __attribute__((aligned(16))) char smem_raw[];
  const int xcd = blockIdx.x % kNumXcd, p = blockIdx.x / kNumXcd, workers = gridDim.x / kNumXcd;
  const int per_group = a.zh_group * a.num_n_tiles;
  const bool ragged = dkdv_level_list<128>(a);
  const int zh_lo = xcd * a.zh_per_xcd;
  LevelWalk walk;
  if (ragged)
    walk.init<256>(reinterpret_cast<uint32_t*>(smem_raw + WideDkDvSmem::BYTES), a.seq, zh_lo,
                   zh_lo + a.zh_per_xcd < a.num_zh ? zh_lo + a.zh_per_xcd : a.num_zh, a.num_zh / a.hk, 1, kWideBN, true,
                   threadIdx.x);
  for (int r = 0; r * workers < a.items_per_xcd; ++r) {
    const int lp = worker_pos<false>(r, p, workers, a.num_cu);
    int zh, nt;
    if (ragged) {
      int e;
      if (!walk.at(lp, e, nt)) break;
      zh = zh_lo + e;
    } else {
      if (lp >= a.items_per_xcd) continue;
      const int gi = lp / per_group, gr = lp % per_group;
      const int zl = gi * a.zh_group + gr % a.zh_group;
      zh = zh_lo + zl;
      if (zl >= a.zh_per_xcd || zh >= a.num_zh) continue;
      nt = gr / a.zh_group;
    }
    int z, hk;
    split_zh(zh, a.num_zh / a.hk, 1, z, hk);
    dkdv_wide_item<T, kWindowed, kPad>(a, hk, nt, z, smem_raw);
    __syncthreads();
  }
}

struct WideDqSmem {
  static constexpr int TILE_BYTES = kWideBM * 128 * 2;
  static constexpr int STAGE_BYTES = 2 * TILE_BYTES;       // K, V (swizzled)
  static constexpr int Q_OFF = STAGE_BYTES;                // the item's Q rows on their way to registers; then stages 1 and 2
  static constexpr int DO_OFF = Q_OFF + kWideBN * 256;     // its dO rows; at the end dQ on its way out
  static constexpr int BYTES = DO_OFF + kWideBN * 256;
  static_assert(3 * STAGE_BYTES <= DO_OFF, "three stages");
};

template <typename T, bool kWindowed, int kPad>
__device__ __forceinline__ void dq_wide_item(const BwdArgs& a, const int h, const int mt, const int z, char* smem_raw) {
  constexpr int D = 128, BM = kWideBN, BN = kWideBM, QB = 2;
  using Tr = Traits<T>;
  using op_t = typename Tr::op_t;
  using q4_t = typename Tr::q4_t;
  using SM = WideDqSmem;
  constexpr int DC = kPad ? kPad : D;
  constexpr int KS = DC / 16, DB = DC / 32, TS = BN / 16, P = TS * DB;      // MFMAs of a pass
  static_assert(KS == P, "one operand slot per MFMA of a pass");
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
  const BlockRanges br = block_ranges(kWindowed, w.left, w.right, q0, si.seqlen_q, si.seqlen_k, BM, BN);
  const int qw = q0 + 64 * wave;
  const BlockRanges wr = block_ranges(kWindowed, w.left, w.right, qw, si.seqlen_q, si.seqlen_k, 64, BN);

  const int hk = h / (a.hq / a.hk);
  const int row0 = qw + c;                       // this lane's queries: row0 and row0 + 32
  const int row4 = lane / 16, ch = lane % 16;
  const int rows_q = si.seqlen_q - qw < 64 ? si.seqlen_q - qw : 64;

  char* area = smem_raw + SM::DO_OFF + wave * 64 * ROWB;
  constexpr int AREA_ROW = 256 + 16;
  T* dq_w = reinterpret_cast<T*>(a.dq) + (int64_t)si.batch_index * a.sdq.z + (int64_t)h * a.sdq.h + (int64_t)(si.q_start + qw) * a.sdq.s;
  auto store_block = [&](int b) __attribute__((always_inline)) {
    const int rows = rows_q - 32 * b;
    const auto rs = wave_rsrc(dq_w + 32 * b * a.sdq.s, rows > 0 ? ((rows - 1) * (int)a.sdq.s + d_qk) * 2 : 0);
    const int voff = ch * 8 < d_qk ? row4 * (int)a.sdq.s * 2 + ch * 16 : kVoffOutOfRange;
#pragma unroll
    for (int i = 0; i < 8; ++i)
      __builtin_amdgcn_raw_buffer_store_b128(*reinterpret_cast<const u32x4_t*>(area + (row4 + 4 * i) * AREA_ROW + ch * 16), rs,
                                             voff, i * 4 * (int)a.sdq.s * 2, 0);
  };

  // ---- the item's Q and dO rows: memory -> LDS -> registers; its O rows for delta
  const int smem0 = lds_offset(smem_raw);
  {
    const T* qp = reinterpret_cast<const T*>(a.q) + (int64_t)si.batch_index * a.sq.z + (int64_t)h * a.sq.h + (int64_t)(si.q_start + qw) * a.sq.s;
    const T* dop = reinterpret_cast<const T*>(a.dout) + (int64_t)si.batch_index * a.sdo.z + (int64_t)h * a.sdo.h + (int64_t)(si.q_start + qw) * a.sdo.s;
    const auto q_rs = wave_rsrc_words(qp, rows_q > 0 ? ((rows_q - 1) * (int)a.sq.s + d_qk) * 2 : 0);
    const auto do_rs = wave_rsrc_words(dop, rows_q > 0 ? ((rows_q - 1) * (int)a.sdo.s + d_v) * 2 : 0);
#pragma unroll
    for (int i = 0; i < 16; i += 2) {
      rows_to_lds(q_rs, row4 * (int)a.sq.s * 2, 4 * (int)a.sq.s * 2, d_qk, smem0 + SM::Q_OFF + wave * 64 * ROWB, i);
      rows_to_lds(do_rs, row4 * (int)a.sdo.s * 2, 4 * (int)a.sdo.s * 2, d_v, smem0 + SM::DO_OFF + wave * 64 * ROWB, i);
    }
  }
  int row_c[QB];
#pragma unroll
  for (int b = 0; b < QB; ++b) row_c[b] = row0 + 32 * b < si.seqlen_q ? row0 + 32 * b : si.seqlen_q - 1;

  // K and V tiles of 32 keys, staged as the dK/dV item stages its Q and dO
  const int ntk = br.lo <= br.hi ? br.hi - br.lo + 1 : 0;
  const int r0 = tid / 16, gch = ch ^ Swz<D>::f(r0);
  const int k_voff = gch * 8 < d_qk ? r0 * (int)a.sk.s * 2 + gch * 16 : kVoffOutOfRange;
  const int v_voff = gch * 8 < d_v ? r0 * (int)a.sv.s * 2 + gch * 16 : kVoffOutOfRange;
  const int k_row = (int)a.sk.s * 2, v_row = (int)a.sv.s * 2;
  const T* kb = reinterpret_cast<const T*>(a.k) + (int64_t)si.batch_index * a.sk.z + (int64_t)hk * a.sk.h + ((int64_t)si.k_start + (int64_t)br.lo * BN) * a.sk.s;
  const T* vb = reinterpret_cast<const T*>(a.v) + (int64_t)si.batch_index * a.sv.z + (int64_t)hk * a.sv.h + ((int64_t)si.k_start + (int64_t)br.lo * BN) * a.sv.s;
  int f_tiles = ntk, f_rows = si.seqlen_k - br.lo * BN;
  u32x4_t k_rs, v_rs;
  auto fetch_begin = [&]() __attribute__((always_inline)) {
    const int rows = f_tiles > 0 ? min(f_rows, BN) : 0;
    k_rs = wave_rsrc_words(kb, rows_extent(rows, k_row, d_qk * 2));
    v_rs = wave_rsrc_words(vb, rows_extent(rows, v_row, d_v * 2));
    kb += (int64_t)BN * a.sk.s; vb += (int64_t)BN * a.sv.s;
    f_rows -= BN; --f_tiles;
  };
  auto fetch_piece = [&](int stage, int i) __attribute__((always_inline)) {
    const int lds = smem0 + stage + i * SM::TILE_BYTES + wave * 4 * ROWB;
    if (i == 0) load_to_lds(k_rs, k_voff, 0, lds, k_voff, 16 * k_row, lds + 16 * ROWB);
    else load_to_lds(v_rs, v_voff, 0, lds, v_voff, 16 * v_row, lds + 16 * ROWB);
  };
  auto fetch_all = [&](int stage) __attribute__((always_inline)) {
    fetch_begin();
#pragma unroll
    for (int i = 0; i < 2; ++i) fetch_piece(stage, i);
  };
  fetch_all(0);

  float l_row[QB], d_row[QB];
  const int64_t st0 = lse_offset(si, h, a.hq);
  op_t qreg[QB][KS], doreg[QB][KS];
  {
    op_t o8[QB][KS];
#pragma unroll
    for (int b = 0; b < QB; ++b) {
      l_row[b] = a.lse[st0 + row_c[b]] * -kRcpLn2;
      const T* optr = reinterpret_cast<const T*>(a.out) + (int64_t)si.batch_index * a.so.z + (int64_t)h * a.so.h + (int64_t)(si.q_start + row_c[b]) * a.so.s;
#pragma unroll
      for (int k = 0; k < KS; ++k) {
        const op_t zero8 = {0, 0, 0, 0, 0, 0, 0, 0};
        o8[b][k] = 16 * k + 8 * hi < d_v ? *reinterpret_cast<const op_t*>(optr + 16 * k + 8 * hi) : zero8;
      }
    }
    const int row_a = Swz<D>::row_base(lane);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    const char* Qt = smem_raw + SM::Q_OFF + wave * 64 * ROWB;
    const char* dOt = smem_raw + SM::DO_OFF + wave * 64 * ROWB;
#pragma unroll
    for (int b = 0; b < QB; ++b) {
#pragma unroll
      for (int k = 0; k < KS; ++k) {
        qreg[b][k] = swz_read_row<T, D>(Qt, row_a, k, b);
        doreg[b][k] = swz_read_row<T, D>(dOt, row_a, k, b);
      }
    }
#pragma unroll
    for (int b = 0; b < QB; ++b) {
      float acc = 0.f;
#pragma unroll
      for (int k = 0; k < KS; ++k)
#pragma unroll
        for (int e = 0; e < 8; ++e) acc += (float)o8[b][k][e] * (float)doreg[b][k][e];
      d_row[b] = cross_sum(acc);
      if (row0 + 32 * b < si.seqlen_q && hi == 0) a.delta[st0 + row0 + 32 * b] = d_row[b];
    }
  }
#pragma unroll
  for (int b = 0; b < QB; ++b)
#pragma unroll
    for (int k = 0; k < KS; ++k) {
      asm volatile("" : "+a"(qreg[b][k]));
      asm volatile("" : "+a"(doreg[b][k]));
    }
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");      // tile 0 is there, Q has left its area

  if (ntk == 0) {      // no key sees these queries
#pragma unroll
    for (int i = 0; i < 8; ++i) *reinterpret_cast<u32x4_t*>(area + (row4 + 4 * i) * AREA_ROW + ch * 16) = u32x4_t{0, 0, 0, 0};
#pragma unroll
    for (int b = 0; b < QB; ++b) store_block(b);
    return;
  }

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

  f32x16 dq[QB][DB];
#pragma unroll
  for (int b = 0; b < QB; ++b)
#pragma unroll
    for (int db = 0; db < DB; ++db) acc_zero<T>(dq[b][db]);

  int st_cur = 0, st_nxt = SM::STAGE_BYTES, st_fetch = 2 * SM::STAGE_BYTES;
  fetch_all(st_nxt);

  const float qk_scale = a.sm_scale * kLog2e;
  const f32x16 zero16 = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  f32x16 nd[QB];
#pragma unroll
  for (int b = 0; b < QB; ++b)
#pragma unroll
    for (int i = 0; i < 16; ++i) nd[b][i] = -d_row[b];

  int ra[KS], tr[2][DB];
  {
    const int row_a = Swz<D>::row_base(lane), tr_a0 = Swz<D>::tr_base(lane, 0), tr_a1 = Swz<D>::tr_base(lane, 1);
#pragma unroll
    for (int k = 0; k < KS; ++k) ra[k] = smem0 + (row_a ^ (k << 5));
#pragma unroll
    for (int db = 0; db < DB; ++db) { tr[0][db] = smem0 + (tr_a0 ^ (db << 6)); tr[1][db] = smem0 + (tr_a1 ^ (db << 6)); }
  }
  auto rotate = [&]() __attribute__((always_inline)) {
    const int step = st_nxt - st_cur, t = st_cur;
#pragma unroll
    for (int k = 0; k < KS; ++k) { ra[k] += step; asm("" : "+v"(ra[k])); }
#pragma unroll
    for (int db = 0; db < DB; ++db) {
      tr[0][db] += step; asm("" : "+v"(tr[0][db]));
      tr[1][db] += step; asm("" : "+v"(tr[1][db]));
    }
    st_cur = st_nxt; st_nxt = st_fetch; st_fetch = t;
  };
  // Operand slots: every operand serves both blocks of queries, in two passes of P MFMAs one after the other; the second pass
  // hands each slot to the operand that is needed a pass later: K rows (S) -> V rows (dP) -> K^T (dQ) -> the next tile's K rows.
  op_t x[P];
  auto k_row_read = [&](int k) __attribute__((always_inline)) { return lds_read<op_t>(ra[k]); };
  auto v_row_read = [&](int k) __attribute__((always_inline)) { return lds_read<op_t>(ra[k] + SM::TILE_BYTES); };
  auto kt_read = [&](int i) __attribute__((always_inline)) {
    const int off = i / DB * 16 * ROWB;
    const q4_t lo = __builtin_bit_cast(q4_t, lds_read_tr_at(tr[0][i % DB] + off));
    const q4_t hi4 = __builtin_bit_cast(q4_t, lds_read_tr_at(tr[1][i % DB] + off));
    return __builtin_shufflevector(lo, hi4, 0, 1, 2, 3, 4, 5, 6, 7);
  };
#pragma unroll
  for (int k = 0; k < P; ++k) x[k] = k_row_read(k);

  auto compute = [&](auto masked_tag, int j) __attribute__((always_inline)) {
    constexpr bool masked = decltype(masked_tag)::value;
    f32x16 s[QB], dp[QB];
    op_t sb[QB][TS];
    unsigned m_d[QB];
#pragma unroll
    for (int b = 0; b < QB; ++b) m_d[b] = m_none[b] ? 0x40000000u : (unsigned)(j * BN + 4 * hi - m_lo[b]);
    auto p_el = [&](int b, int i) __attribute__((always_inline)) {
      float v = __builtin_fmaf(s[b][i], qk_scale, l_row[b]);
      if (masked) {
        const bool vis = m_d[b] + (unsigned)(8 * (i / 4) + i % 4) <= m_rng[b];
        v = vis ? v : -__builtin_inff();
      }
      s[b][i] = fast_exp2(v);
    };
    auto ds_el = [&](int b, int i) __attribute__((always_inline)) {
      dp[b][i] = s[b][i] * dp[b][i];      // (dP started at -delta)
      if (i & 1) {
        const typename Tr::p2_t s2 = Tr::cvt2(dp[b][i - 1], dp[b][i]);
        sb[b][i / 8][i % 8 - 1] = s2[0];
        sb[b][i / 8][i % 8] = s2[1];
      }
    };
    // the vector work, spread over the MFMAs between the one that makes its input and the one that needs its result: slot i
    // is the i-th of the tile's 6 P MFMAs (S of block 0, S of block 1, dP, dP, dQ, dQ)
    auto work = [&](int slot) __attribute__((always_inline)) {
      auto span = [&](int from, int to, auto f) __attribute__((always_inline)) {
        if (slot < from || slot >= to) return;
#pragma unroll
        for (int i = first_of(slot - from, 16, to - from); i < first_of(slot + 1 - from, 16, to - from); ++i) f(i);
      };
      span(P + 1, 2 * P + P / 2, [&](int i) __attribute__((always_inline)) { p_el(0, i); });
      span(2 * P + P / 2, 4 * P - 2, [&](int i) __attribute__((always_inline)) { p_el(1, i); });
      span(3 * P + 1, 4 * P + P / 2 - 2, [&](int i) __attribute__((always_inline)) { ds_el(0, i); });
      span(4 * P + 1, 5 * P + P / 2 - 2, [&](int i) __attribute__((always_inline)) { ds_el(1, i); });
      __builtin_amdgcn_sched_barrier(0);
    };
#pragma unroll
    for (int i = 0; i < P; ++i) {
      s[0] = Tr::mfma(x[i], qreg[0][i], i == 0 ? zero16 : s[0]);
      work(i);
    }
#pragma unroll
    for (int i = 0; i < P; ++i) {
      s[1] = Tr::mfma(x[i], qreg[1][i], i == 0 ? zero16 : s[1]);
      x[i] = v_row_read(i);
      work(P + i);
    }
#pragma unroll
    for (int i = 0; i < P; ++i) {
      dp[0] = Tr::mfma(x[i], doreg[0][i], i == 0 ? nd[0] : dp[0]);
      work(2 * P + i);
    }
#pragma unroll
    for (int i = 0; i < P; ++i) {
      dp[1] = Tr::mfma(x[i], doreg[1][i], i == 0 ? nd[1] : dp[1]);
      x[i] = kt_read(i);
      work(3 * P + i);
    }
#pragma unroll
    for (int i = 0; i < P; ++i) {
      mfma_acc<T>(dq[0][i % DB], x[i], sb[0][i / DB]);
      work(4 * P + i);
    }
    // the next tile has landed (requested a tile ago), and every wave has left the tile before this one
    asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier\n\ts_nop 1" ::: "memory");
    rotate();
    fetch_begin();
#pragma unroll
    for (int i = 0; i < P; ++i) {
      mfma_acc<T>(dq[1][i % DB], x[i], sb[1][i / DB]);
      x[i] = k_row_read(i);
      if (i == 0 || i == 2) fetch_piece(st_nxt, i / 2);
      work(5 * P + i);
    }
  };
  auto skip = [&]() __attribute__((always_inline)) {
    asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
    rotate();
    fetch_all(st_nxt);
#pragma unroll
    for (int k = 0; k < P; ++k) x[k] = k_row_read(k);
  };
  const bool none = wr.lo > wr.hi, full = !none && wr.fb_lo <= wr.fb_hi;
  const int j_lo = none ? br.hi + 1 : wr.lo, j_end = none ? br.hi + 1 : wr.hi + 1;
  const int f_lo = full ? wr.fb_lo : j_end, f_end = full ? wr.fb_hi + 1 : j_end;
  int j = br.lo;
  for (; j < j_lo; ++j) skip();
  for (; j < f_lo; ++j) compute(std::true_type{}, j);
  for (; j < f_end; ++j) compute(std::false_type{}, j);
  for (; j < j_end; ++j) compute(std::true_type{}, j);
  for (; j <= br.hi; ++j) skip();
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  acc_settle(dq[0], dq[1]);
#pragma unroll
  for (int b = 0; b < QB; ++b) {
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        q4_t t4;
#pragma unroll
        for (int r = 0; r < 4; ++r) t4[r] = Tr::cvt(dq[b][db][4 * g + r] * a.sm_scale);
        *reinterpret_cast<q4_t*>(area + c * AREA_ROW + (32 * db + 8 * g + 4 * hi) * 2) = t4;
      }
    __builtin_amdgcn_sched_barrier(0);
    store_block(b);
    __builtin_amdgcn_sched_barrier(0);
  }
}

template <typename T, bool kWindowed, int kPad>
__global__ __attribute__((amdgpu_flat_work_group_size(256, 256))) __attribute__((amdgpu_waves_per_eu(1, 1)))
void bwd_dq_wide_kernel(const BwdArgs a) {
  extern __shared__ __attribute__((aligned(16))) char smem_raw[];
  const int xcd = blockIdx.x % kNumXcd, p = blockIdx.x / kNumXcd, workers = gridDim.x / kNumXcd;
  const int per_group = a.zh_group * a.num_m_tiles;
  // Sequences of different lengths: the valid tiles only, by their distance from the start of the sequence, which is their
  // weight under a causal mask (16 packed sequences of 256-8192 tokens, Hq 32 Hk 8: 4760 -> 4250 us against the dense list).
  const bool ragged = a.seq.num_seqlens != 0 && a.zh_per_xcd <= kLevelCap && a.num_m_tiles <= 0xffff;
  const int zh_lo = xcd * a.zh_per_xcd;
  LevelWalk walk;
  if (ragged)
    walk.init<256>(reinterpret_cast<uint32_t*>(smem_raw + WideDqSmem::BYTES), a.seq, zh_lo,
                   zh_lo + a.zh_per_xcd < a.num_zh ? zh_lo + a.zh_per_xcd : a.num_zh, a.num_zh / a.hq, a.hq / a.hk, kWideBN,
                   false, threadIdx.x);
  for (int r = 0; r * workers < a.items_per_xcd; ++r) {
    const int li = worker_pos<false>(r, p, workers, a.num_cu);
    int zh, mt;
    if (ragged) {
      int e;
      if (!walk.at(li, e, mt)) break;
      zh = zh_lo + e;
    } else {
      if (li >= a.items_per_xcd) continue;
      const int gi = li / per_group, gr = li % per_group;
      const int zl = gi * a.zh_group + gr % a.zh_group;
      zh = zh_lo + zl;
      if (zl >= a.zh_per_xcd || zh >= a.num_zh) continue;
      mt = a.num_m_tiles - 1 - gr / a.zh_group;
    }
    int z, h;
    split_zh(zh, a.num_zh / a.hq, a.hq / a.hk, z, h);
    dq_wide_item<T, kWindowed, kPad>(a, h, mt, z, smem_raw);
    __syncthreads();
  }
}

template <typename T, bool W, int kPad>
hipError_t launch_dq_wide(const BwdArgs& a0, hipStream_t stream) {
  BwdArgs a = a0;
  a.num_m_tiles = (a.seq.max_seqlen_q + kWideBN - 1) / kWideBN;
  set_work(a, tile_work(bwd_nseq(a) * a.hq, a.walk_group, a.num_m_tiles));
  dim3 grid((unsigned)(kNumXcd * bwd_workers(128, false, a.items_per_xcd, a.num_cu, 1)));
  return launch_with_lds<bwd_dq_wide_kernel<T, W, kPad>>(grid, 256, WideDqSmem::BYTES + kLevelBytes, stream, a);
}

template <typename T, bool W, int kPad>
hipError_t launch_dkdv_wide(const BwdArgs& a0, hipStream_t stream) {
  BwdArgs a = a0;
  a.num_n_tiles = (a.seq.max_seqlen_k + kWideBN - 1) / kWideBN;
  set_work(a, tile_work(bwd_nseq(a) * a.hk, a.walk_group, a.num_n_tiles));
  dim3 grid((unsigned)(kNumXcd * bwd_workers(128, false, a.items_per_xcd, a.num_cu, 1)));
  return launch_with_lds<bwd_dkdv_wide_kernel<T, W, kPad>>(grid, 256, WideDkDvSmem::BYTES + kLevelBytes, stream, a);
}

}  // namespace fa
