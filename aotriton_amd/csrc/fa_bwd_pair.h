// dK, dV (and the stored dS) by pairs of waves: the dK/dV kernel of the backward that keeps dS (fa_bwd_impl.h, BwdArgs::ds_ws)
// at head dims above 128, for 16-bit types, dense batches, no bias or a plain one (plain_bias).
//
// A workgroup owns 128 keys of one kv-head on eight waves, two per SIMD.  The two waves of a 32-key block share its work by
// product instead of by rows:
//   wave w      S = Q K^T, P = exp2(..) with bias, mask and dropout | dV^T += dO^T P                       holds K and dV
//   wave w + 4  dP = dO V^T                                         | dS = P (dP - delta), dK^T += Q^T dS  holds V and dK, stores dS
// P travels from one to the other through LDS in fp32 as it lies in the lanes (both products have the same layout); its sign says
// whether dropout keeps the element.  Nothing is computed twice and no sum changes its order: the results are those of dkdv_item.
//
// Why: a wave that does all four products of its keys needs more than 256 registers at D = 256 (dK, dV, K and half a V), runs alone
// on its SIMD and issues MFMAs, vector and LDS instructions one after the other.  Half of each fits 256, so that one wave's
// exponentials and Philox rounds stand next to the other's MFMAs.
//
// A step is 32 queries and has a barrier in its middle (P is there) and one at its end.  Q, dO, the row statistics and a bias go
// straight into LDS two steps ahead of their use; the first waves request all of it, so that a wait for vector memory never waits for
// the second waves' stores of dS.  What the loop must not have is a wait that the compiler adds: a spilled register's reload, or loads
// from in front of the loop that it takes to be under way, cost 5-15 % each here.
//
// Measured, us, dkdv_item -> this, one card each: window 1024, bias and dropout, B2 H16 S8192 fp16, this kernel 975 -> 811 (matrix pipe
// 29 -> 37 % busy, vector ALU 36 -> 45 %, at 1.85-1.95 GHz; what is left is that the two waves of a SIMD want the same unit in turn, and the barriers),
// forward and backward 1831 -> 1713; backward alone, bf16: B2 H16 S4096 causal 790 -> 750, Hq 32 Hk 8 S1000 202 -> 191, D200 S2048 causal 243 -> 222.
// 128 columns: level (B4 H16 1000 x 1531 with dropout 313 / 314, window, bias and dropout S2048 186 / 182, B1 Hq 32 Hk 8 S1024 110 / 113); a bias with rows
// anywhere: 2 % slower, its pieces pass through registers.
#pragma once
#include "fa_bwd_impl.h"
#include "fa_wide.h"

namespace fa {

template <bool kBias>
struct PairSmem {
  static constexpr int D = 256;
  static constexpr int BM = 32, BN = 128;
  static constexpr int STAGES = 3;
  static constexpr int TILE_BYTES = BM * D * 2;
  static constexpr int STAT_BYTES = 1024;      // what one wave instruction fills: L and delta as prepared, BM floats each, and nothing
  static constexpr int STAGE_BYTES = 2 * TILE_BYTES + STAT_BYTES;      // Q, dO (swizzled), statistics
  static constexpr int BIAS_OFF = STAGES * STAGE_BYTES, BIAS_BYTES = BM * BN * 2;      // rows of 128 keys, swizzled like a tile of 128 columns
  static constexpr int P_OFF = BIAS_OFF + (kBias ? STAGES * BIAS_BYTES : 0), P_BYTES = 4 * 32 * BM * 4;
  static constexpr int KW_OFF = P_OFF + P_BYTES;      // keep bits, a word per lane of the first waves
  // The last k-steps' operands of the eight waves' own rows, for which there are no registers (a spilled one's reload waits for all
  // vector memory in flight).
  static constexpr int OWN = kBias ? 2 : 4, OWN_OFF = KW_OFF + 4 * 64 * 4;
  static constexpr int BYTES = OWN_OFF + 8 * OWN * 1024;
  static_assert(STAGE_BYTES % 512 == 0 && TILE_BYTES % 512 == 0, "stage offsets leave the swizzled bits alone");
};

// The lane's number, formed where it is used: what is derived from it then does not stay in registers over the steps.
__device__ __forceinline__ int lane_here() {
  int x;
  asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(x));
  return x;
}

template <typename T, bool kWindowed, bool kBias, bool kDropout, int kPad>
__device__ __forceinline__ void dkdv_pair_item(const BwdArgs& a, const int hk, const int nt, const int z, const int part,
                                               char* smem_raw) {
  using Tr = Traits<T>;
  using op_t = typename Tr::op_t;
  using q4_t = typename Tr::q4_t;
  using SM = PairSmem<kBias>;
  constexpr int D = SM::D, BM = SM::BM, BN = SM::BN;
  using DT = DsTile<T, D>;
  static_assert(BM == DT::BM && BN == DT::BN, "stored tiles have the item's shape");
  constexpr int DC = kPad ? kPad : D;            // columns computed; those past a tensor's head dim are zero
  constexpr int KS = DC / 16, DB = DC / 32, TS = BM / 16, G = TS * DB;
  constexpr int LPR = D / 8, RPI = 256 / LPR, RWI = 64 / LPR, CH = BM / RPI;      // 16-byte chunks per row; rows per access of four waves, of one; accesses per tile
  constexpr int ROWB = Swz<D>::ROWB;
  static_assert(RPI % 8 == 0 && CH % 2 == 0, "the swizzle repeats every two accesses");

  const int lane = threadIdx.x & 63, c = lane & 31, hi = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int w = wave & 3;                        // key block
  const bool first = wave < 4;
  const int d_qk = kPad ? a.head_dim : D, d_v = kPad ? a.head_dim_v : D;

  const SeqInfo si = get_seq(a.seq, z);
  const int n0 = nt * BN;
  if (n0 >= si.seqlen_k) return;

  Window win{0, 0};
  if (kWindowed) win = parse_window(a.mask.causal_type, a.mask.window_left, a.mask.window_right, si.seqlen_q, si.seqlen_k);
  win.left = win.left > (1 << 30) ? (1 << 30) : (win.left < -(1 << 30) ? -(1 << 30) : win.left);
  win.right = win.right > (1 << 30) ? (1 << 30) : (win.right < -(1 << 30) ? -(1 << 30) : win.right);
  BlockRanges br = block_ranges(kWindowed, win.right, win.left, n0, si.seqlen_k, si.seqlen_q, BN, BM);

  const int group = a.hq / a.hk;
  int g_lo = 0, g_hi = group;
  float* part_ptr = nullptr;      // this part's fp32 sums, where items are cut
  if (a.part_ws != nullptr) {
    const int ph = part / a.part_tiles, pt = part % a.part_tiles, hs = group / a.part_heads;
    g_lo = ph * hs;
    g_hi = g_lo + hs;
    const int per = (br.hi - br.lo + a.part_tiles) / a.part_tiles;
    br.lo += pt * per;
    if (br.lo + per - 1 < br.hi) br.hi = br.lo + per - 1;
    part_ptr = a.part_ws + (((int64_t)(z * a.hk + hk) * a.num_n_tiles + nt) * (a.part_heads * a.part_tiles) + part) * (2 * BN * D) +
               (first ? BN * D : 0);
  }

  const int key = n0 + w * 32 + c;
  const bool key_ok = key < si.seqlen_k;
  const int key_c = key_ok ? key : si.seqlen_k - 1;

  f32x16 acc[DB];                                // dV^T or dK^T of the wave's keys
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[db][i] = 0.f;
  auto finish = [&](float scale) {
    const int x = lane_here(), c = x & 31, hi = x >> 5, key = n0 + w * 32 + c;
    if (part_ptr != nullptr) {
      float* p = part_ptr + (w * 32 + c) * D + 4 * hi;
#pragma unroll
      for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int g = 0; g < 4; ++g)
          *reinterpret_cast<f32x4*>(p + 32 * db + 8 * g) = f32x4{acc[db][4 * g], acc[db][4 * g + 1], acc[db][4 * g + 2], acc[db][4 * g + 3]};
      return;
    }
    if (key >= si.seqlen_k) return;
    const KernelArgs<BwdArgs> k = kernel_args<BwdArgs>();
    T* const out = first ? reinterpret_cast<T*>(k->dv) + (int64_t)si.batch_index * k->sdv.z + (int64_t)hk * k->sdv.h + (int64_t)(si.k_start + key) * k->sdv.s
                         : reinterpret_cast<T*>(k->dk) + (int64_t)si.batch_index * k->sdk.z + (int64_t)hk * k->sdk.h + (int64_t)(si.k_start + key) * k->sdk.s;
    const int d_out = first ? d_v : d_qk;        // columns of this wave's result
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        q4_t x;
#pragma unroll
        for (int r = 0; r < 4; ++r) x[r] = Tr::cvt(acc[db][4 * g + r] * scale);      // bwd_kernel_dk_dv.py:387-389
        if (32 * db + 8 * g + 4 * hi < d_out) *reinterpret_cast<q4_t*>(out + 32 * db + 8 * g + 4 * hi) = x;
      }
  };
  if (br.lo > br.hi) {      // no query (of this part) sees these keys
    finish(1.0f);
    return;
  }

  // this lane's key row of K or V, an operand with k = head dim
  constexpr int KO = SM::OWN, KR = KS - KO;      // k-steps whose operands are in LDS, in registers
  op_t own[KR];
  auto own_place = [&](int lane) { return lds_offset(smem_raw) + SM::OWN_OFF + wave * (KO * 1024) + lane * 16; };
  {
    const int own_at = own_place(lane);
    const T* row = first ? reinterpret_cast<const T*>(a.k) + (int64_t)si.batch_index * a.sk.z + (int64_t)hk * a.sk.h + (int64_t)(si.k_start + key_c) * a.sk.s
                         : reinterpret_cast<const T*>(a.v) + (int64_t)si.batch_index * a.sv.z + (int64_t)hk * a.sv.h + (int64_t)(si.k_start + key_c) * a.sv.s;
    const int d_in = first ? d_qk : d_v;
    const op_t zero8 = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
    for (int k = 0; k < KS; ++k) {
      const op_t x = 16 * k + 8 * hi < d_in ? *reinterpret_cast<const op_t*>(row + 16 * k + 8 * hi) : zero8;
      if (k < KR) own[k] = x;
      else lds_write(own_at + (k - KR) * 1024, x);
    }
  }

  // In front of the steps: the compiler otherwise waits in every one of them for the loads that brought `own`, and with them for
  // whatever else is in flight.  (vmcnt 0; the other counters stay as they are)
  auto own_here = [&]() { __builtin_amdgcn_s_waitcnt(0x0F70); };
  const int ntq = br.hi - br.lo + 1;     // steps per q-head
  const int smem0 = lds_offset(smem_raw);
  // LDS addresses of the running stage's operands.  The swizzle moves 16-byte chunks inside 256 bytes, so what picks an operand is
  // one exclusive or with the lane's base; the rest is an offset of the instruction.  (Eight rows on, the chunks of a transposing
  // read lie two positions apart, which is bit 5.)
  int row_at = smem0 + Swz<D>::row_base(lane), tr_at = smem0 + Swz<D>::tr_base(lane, 0), stat_at = smem0 + 2 * SM::TILE_BYTES + 16 * hi;
  int stage = 0;
  auto next_stage = [&]() {
    const int d = stage == SM::STAGES - 1 ? (1 - SM::STAGES) * SM::STAGE_BYTES : SM::STAGE_BYTES;
    stage = stage == SM::STAGES - 1 ? 0 : stage + 1;
    row_at += d; tr_at += d; stat_at += d;
  };
  auto read_row = [&](int tile, int k) { return lds_read<op_t>((row_at ^ ((k & 7) << 5)) + (tile + (k >> 3) * 256)); };
  auto read_tr = [&](int tile, int i) {
    const int t = i / DB, db = i % DB, off = tile + t * 16 * ROWB + (db >> 2) * 256;
    const q4_t x = __builtin_bit_cast(q4_t, lds_read_tr_at((tr_at ^ ((db & 3) << 6)) + off));
    const q4_t y = __builtin_bit_cast(q4_t, lds_read_tr_at((tr_at ^ ((db & 3) << 6 | 32)) + (off + 8 * ROWB)));
    return __builtin_shufflevector(x, y, 0, 1, 2, 3, 4, 5, 6, 7);
  };
  auto read_stat = [&](int which, int g) { return lds_read<f32x4>(stat_at + which * BM * 4 + 32 * g); };
  auto p_place = [&](int lane) { return smem0 + SM::P_OFF + w * 4096 + lane * 16; };
  auto kw_place = [&](int lane) { return smem0 + SM::KW_OFF + w * 256 + lane * 4; };
  const f32x16 zero16 = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};

  // ---- keep bits, a step ahead: a Philox call yields those of four consecutive keys, the four lanes of a quad, for one row; quad
  // lane q runs the calls of the rows with m % 4 == q (see dkdv_item), four a step.  The first waves run kOwn of them behind their dV, the
  // second waves the others behind their dP.
    constexpr int kOwn = 2;
  const uint32_t own_rows = first ? 0 : 8 * kOwn;
  uint64_t ctr = 0;                              // of this lane's first call of the step
  uint32_t x_stride = 0, x_k0 = 0, x_k1 = 0;
  int32_t x_thr = 0;
  int x_left = 0, x_g = g_lo;                    // steps left of the head, the next head
  Philox px;
  uint32_t word = 0;
  auto keep_begin = [&]() {
    if (x_left == 0 && x_g < g_hi) {
      const KernelArgs<BwdArgs> k = kernel_args<BwdArgs>();
      DropoutArgs d;
      d.p = k->drop.p; d.seed_ptr = k->drop.seed_ptr; d.offset1_ptr = k->drop.offset1_ptr; d.offset2 = k->drop.offset2;
      const DropoutState s = dropout_for_head(make_dropout_base(d, k->seq.max_seqlen_k), z, hk * group + x_g++, k->hq, k->seq.max_seqlen_q);
      x_stride = __builtin_amdgcn_readfirstlane(s.stride);
      x_k0 = __builtin_amdgcn_readfirstlane(s.k0);
      x_k1 = __builtin_amdgcn_readfirstlane(s.k1);
      x_thr = __builtin_amdgcn_readfirstlane(s.thr);
      x_left = ntq;
      const int x = lane_here();
      ctr = s.base + (uint64_t)(br.lo * BM + own_rows + 4 * (x >> 5) + (x & 3)) * s.stride + (uint64_t)((n0 + w * 32 + (x & 31)) >> 2);
    }
    --x_left;
    word = 0;
  };
  auto keep_end = [&]() { ctr += 32ull * x_stride; };
  auto keep_round = [&](int i) __attribute__((always_inline)) {      // round i % 10 of call i / 10
    if (i % 10 == 0) {
      const uint64_t at = ctr + (uint64_t)(8 * (i / 10)) * x_stride;
      px.start((uint32_t)at, (uint32_t)(at >> 32));
    }
    px.round(i % 10, x_k0, x_k1);
    if (i % 10 == 9) word = dropout_append(px, x_thr, word);
  };
  constexpr int kRows = 4, kRing = 4;        // operands in flight: rows, transposed

  if (first) {
    __builtin_amdgcn_s_setprio(2);                 // (theirs is the longer way to P)
    // ---- staging: Q, dO, the statistics and the bias of the step after the next ------------------
    const int tid = threadIdx.x;                 // (of the four first waves)
    const int r0 = tid / LPR, cc0 = tid % LPR;
    int q_voff[2], do_voff[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const int gch = cc0 ^ Swz<D>::f(r0 + k * RPI);
      q_voff[k] = gch * 8 < d_qk ? r0 * (int)a.sq.s * 2 + gch * 16 : kVoffOutOfRange;
      do_voff[k] = gch * 8 < d_v ? r0 * (int)a.sdo.s * 2 + gch * 16 : kVoffOutOfRange;
    }
    const int q_row = own_scalar((int)a.sq.s * 2), do_row = own_scalar((int)a.sdo.s * 2), bias_row = kBias ? own_scalar((int)a.sb_m * 2) : 0;
    const int b_voff = kBias ? tid / 16 * bias_row + (tid % 16 ^ Swz<128>::f(tid / 16)) * 16 : 0;      // of a bias tile (and 16 rows on)
    const int b_cols = si.seqlen_k - n0 < BN ? si.seqlen_k - n0 : BN;
    // lanes 0-7 fetch L, 8-15 delta, which lies behind it in the workspace
    const int st_apart = own_scalar((int)((const char*)a.delta_prep - (const char*)a.lse_scaled));
    const int st_voff = lane < 8 ? lane * 16 : lane < 16 ? st_apart + (lane - 8) * 16 : kVoffOutOfRange;
    const char* qb = nullptr; const char* dob = nullptr; const char* bb = nullptr;
    const float* lse_b = nullptr;
    int f_left = 0, f_g = g_lo, f_m = 0;         // steps left of the head being fetched, the next head, first query
    u32x4_t q_rs, do_rs, b_rs, l_rs;
    auto fetch_begin = [&]() {
      if (f_left == 0 && f_g < g_hi) {
        const KernelArgs<BwdArgs> k = kernel_args<BwdArgs>();
        const int hq = hk * group + f_g++;
        f_left = ntq;
        f_m = br.lo * BM;
        const int64_t row0 = (int64_t)si.q_start + f_m;
        qb = reinterpret_cast<const char*>(k->q) + ((int64_t)si.batch_index * k->sq.z + (int64_t)hq * k->sq.h + row0 * k->sq.s) * 2;
        dob = reinterpret_cast<const char*>(k->dout) + ((int64_t)si.batch_index * k->sdo.z + (int64_t)hq * k->sdo.h + row0 * k->sdo.s) * 2;
        lse_b = k->lse_scaled + lse_offset(si, hq, k->hq) + f_m;
        if (kBias)
          bb = reinterpret_cast<const char*>(k->bias) +
               ((int64_t)si.batch_index * k->sb_z + (int64_t)hq * k->sb_h + (int64_t)f_m * k->sb_m + n0) * 2;
      }
      int rows = si.seqlen_q - f_m;
      rows = rows < BM ? rows : BM;
      rows = f_left > 0 && rows > 0 ? rows : 0;
      q_rs = wave_rsrc_words(qb, rows_extent(rows, q_row, d_qk * 2));
      do_rs = wave_rsrc_words(dob, rows_extent(rows, do_row, d_v * 2));
      l_rs = wave_rsrc_words(lse_b, rows > 0 ? st_apart + rows * 4 : 0);
      if (kBias) b_rs = wave_rsrc_words(bb, rows_extent(rows, bias_row, b_cols * 2));
    };
    constexpr int PIECES = CH + (kBias ? 2 : 1), LOADS = 2 * CH + 1 + (kBias ? 2 : 0);      // (loads into LDS)
    int f_at = smem0 + w * RWI * ROWB, f_st = smem0 + 2 * SM::TILE_BYTES, f_b = smem0 + SM::BIAS_OFF, f_stage = 0;      // places being filled
    int b_at = smem0 + SM::BIAS_OFF + (Swz<128>::tr_base(lane, 0) ^ (w << 6));      // this lane's of the bias tile being read
    auto fetch_piece = [&](int i) {
      if (i < CH / 2) {
        load_to_lds(q_rs, q_voff[0], 2 * i * RPI * q_row, f_at + 2 * i * RPI * ROWB, q_voff[1], (2 * i + 1) * RPI * q_row,
                    f_at + (2 * i + 1) * RPI * ROWB);
      } else if (i < CH) {
        const int k = 2 * i - CH;
        load_to_lds(do_rs, do_voff[0], k * RPI * do_row, f_at + SM::TILE_BYTES + k * RPI * ROWB, do_voff[1], (k + 1) * RPI * do_row,
                    f_at + SM::TILE_BYTES + (k + 1) * RPI * ROWB);
      } else if (i == CH) {
        load_to_lds1(l_rs, st_voff, f_st);       // (all four waves write the same)
      } else {
        load_to_lds(b_rs, b_voff, 0, f_b + w * 1024, b_voff, 16 * bias_row, f_b + w * 1024 + 4096);
      }
    };
    auto fetch_end = [&]() {
      qb += BM * q_row; dob += BM * do_row; lse_b += BM;
      if (kBias) bb += BM * bias_row;
      f_m += BM;
      --f_left;
      const bool wrap = f_stage == SM::STAGES - 1;
      f_stage = wrap ? 0 : f_stage + 1;
      const int d = wrap ? (1 - SM::STAGES) * SM::STAGE_BYTES : SM::STAGE_BYTES;
      f_at += d; f_st += d;
      f_b += wrap ? (1 - SM::STAGES) * SM::BIAS_BYTES : SM::BIAS_BYTES;
    };

    const float qk_scale = a.sm_scale * kLog2e;
    int q_lo = 0, q_hi = si.seqlen_q - 1;        // queries that see this lane's key
    if (kWindowed) {
      q_lo = key - win.right > 0 ? key - win.right : 0;
      q_hi = key + win.left < q_hi ? key + win.left : q_hi;
    }
    const bool q_none = !key_ok || q_hi < q_lo;
    const unsigned q_rng = q_none ? 0u : (unsigned)(q_hi - q_lo);
    unsigned q_d = q_none ? 0x40000000u : (unsigned)(br.lo * BM + 4 * hi - q_lo);      // this lane's first query of the step from q_lo

    auto step = [&](auto masked_tag) __attribute__((always_inline)) {
      constexpr bool masked = decltype(masked_tag)::value;
      // ---- S = Q K^T
      op_t xa[kRows], ob[2];
      int own_at = 0;
      f32x16 s;
#pragma unroll
      for (int k = 0; k < kRows - 1; ++k) xa[k] = read_row(0, k);
#pragma unroll
      for (int k = 0; k < KS; ++k) {
        if (k + kRows - 1 < KS) xa[(k + kRows - 1) % kRows] = read_row(0, k + kRows - 1);
        if (k + 1 == KR) own_at = own_place(lane_here());
        if (k + 1 >= KR && k + 1 < KS) ob[(k + 1) & 1] = lds_read<op_t>(own_at + (k + 1 - KR) * 1024);
        s = Tr::mfma(xa[k % kRows], k < KR ? own[k < KR ? k : 0] : ob[k & 1], k == 0 ? zero16 : s);
        __builtin_amdgcn_sched_barrier(0);
      }
      // ---- P
      uint32_t kw[4] = {0, 0, 0, 0};
      const int here = lane_here(), p_at = p_place(here);
      if (kDropout) {
        // all keep bits of the quad's row r, the one of this lane's key first of each call's four
        const uint32_t x = word << (16 - 4 * kOwn) | lds_read<uint32_t>(kw_place(here));
        kw[0] = (uint32_t)__builtin_amdgcn_mov_dpp((int)x, 0x00, 0xf, 0xf, true) << (here & 3);
        kw[1] = (uint32_t)__builtin_amdgcn_mov_dpp((int)x, 0x55, 0xf, 0xf, true) << (here & 3);
        kw[2] = (uint32_t)__builtin_amdgcn_mov_dpp((int)x, 0xaa, 0xf, 0xf, true) << (here & 3);
        kw[3] = (uint32_t)__builtin_amdgcn_mov_dpp((int)x, 0xff, 0xf, 0xf, true) << (here & 3);
      }
      f32x4 l4[2];
      q4_t b4[2];
      op_t pb[TS];
      auto bias_read = [&](int g) { return __builtin_bit_cast(q4_t, lds_read_tr_at((g & 1 ? (b_at ^ 32) + 2048 : b_at) + (g >> 1) * 4096)); };
      l4[0] = read_stat(0, 0);
      if (kBias) b4[0] = bias_read(0);
      f32x4 pw;
      float kept[2];
#pragma unroll
      for (int E = 0; E < 16; ++E) {
        const int g = E / 4, r = E % 4;
        if (r == 0 && g < 3) {
          l4[(g + 1) & 1] = read_stat(0, g + 1);
          if (kBias) b4[(g + 1) & 1] = bias_read(g + 1);
        }
        // p = exp2(s c + (bias log2e - L log2e)) (bwd_inner_dk_dv.py:187-188)
        const float l = -l4[g & 1][r];
        float x = __builtin_fmaf(s[E], qk_scale, kBias ? __builtin_fmaf((float)b4[g & 1][r], kLog2e, l) : l);
        if (masked) {
          const bool vis = q_d + (unsigned)(8 * g + r) <= q_rng;
          x = vis ? x : -__builtin_inff();
        }
        const float p = fast_exp2(x);
        if (kDropout) {
          int keep;
          switch (g) {      // the keep bit spread over a register
            case 0: asm("v_bfe_i32 %0, %1, 15, 1" : "=v"(keep) : "v"(kw[r])); break;
            case 1: asm("v_bfe_i32 %0, %1, 11, 1" : "=v"(keep) : "v"(kw[r])); break;
            case 2: asm("v_bfe_i32 %0, %1, 7, 1" : "=v"(keep) : "v"(kw[r])); break;
            default: asm("v_bfe_i32 %0, %1, 3, 1" : "=v"(keep) : "v"(kw[r])); break;
          }
          const int bits = __builtin_bit_cast(int, p);
          kept[E & 1] = __builtin_bit_cast(float, bits & keep);      // :200-201 (the scale is in p)
          pw[r] = __builtin_bit_cast(float, __builtin_amdgcn_bitop3_b32(bits, keep, (int)0x80000000, 0xf2));      // bits | (~keep & sign)
        } else {
          kept[E & 1] = p;
          pw[r] = p;
        }
        if (E & 1) {      // p cast to dO's dtype (composed_tensors.py:191-193)
          const typename Tr::p2_t p2 = Tr::cvt2(kept[0], kept[1]);
          pb[E / 8][E % 8 - 1] = p2[0];
          pb[E / 8][E % 8] = p2[1];
        }
        if (r == 3) lds_write(p_at + g * 1024, pw);
      }
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");      // P is there
      // ---- dV^T += dO^T P, with the requests and the next step's keep bits behind its MFMAs
      if (kDropout) keep_begin();
      op_t ta[kRing];
#pragma unroll
      for (int i = 0; i < kRing - 1; ++i) ta[i] = read_tr(SM::TILE_BYTES, i);
#pragma unroll
      for (int i = 0; i < G; ++i) {
        if (i + kRing - 1 < G) ta[(i + kRing - 1) % kRing] = read_tr(SM::TILE_BYTES, i + kRing - 1);
        acc[i % DB] = Tr::mfma(ta[i % kRing], pb[i / DB], acc[i % DB]);
        if (i == 0) fetch_begin();
        static_assert(PIECES < G, "a request behind each MFMA");
        if (i >= 1 && i <= PIECES) fetch_piece(i - 1);
        if (kDropout)
#pragma unroll
          for (int j = first_of(i, kOwn * 10, G); j < first_of(i + 1, kOwn * 10, G); ++j) keep_round(j);
        __builtin_amdgcn_sched_barrier(0);
      }
      fetch_end();
      if (kDropout) keep_end();
      // What the next step reads has landed (loads arrive in the order of their requests; this step's, for the one after it, may be
      // under way).
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" :: "n"(LOADS) : "memory");
      next_stage();
      if (kBias) b_at += stage == 0 ? (1 - SM::STAGES) * SM::BIAS_BYTES : SM::BIAS_BYTES;
      if (masked || kWindowed) q_d += BM;
    };

    for (int t = 0; t < 2; ++t) {
      fetch_begin();
#pragma unroll
      for (int i = 0; i < PIECES; ++i) fetch_piece(i);
      fetch_end();
    }
    if (kDropout) {
      keep_begin();
#pragma unroll
      for (int i = 0; i < kOwn * 10; ++i) keep_round(i);
      keep_end();
    }
    own_here();
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    // The query tiles of a q-head come as [masked | whole | masked]; keys past the sequence make all of them masked.
    const bool ragged = n0 + BN > si.seqlen_k;
    const int fb_lo = br.fb_lo < br.lo ? br.lo : br.fb_lo, fb_hi = br.fb_hi > br.hi ? br.hi : br.fb_hi;
    const int n_lb = fb_lo <= fb_hi && !ragged ? fb_lo - br.lo : ntq;
    const int n_end = fb_lo <= fb_hi && !ragged ? fb_hi + 1 - br.lo : ntq;
    for (int g = g_lo; g < g_hi; ++g) {
      int e = 0;
      for (; e < n_lb; ++e) step(std::true_type{});
      for (; e < n_end; ++e) step(std::false_type{});
      if (!kWindowed) q_d += (unsigned)(n_end - n_lb) * BM;
      for (; e < ntq; ++e) step(std::true_type{});
      q_d -= (unsigned)ntq * BM;
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");      // (requests past the last step)
    finish(1.0f);
  } else {
    constexpr int kDsStorePolicy = 2 | 16;       // as dkdv_item's
    char* ds_tile = nullptr;
    auto step = [&]() __attribute__((always_inline)) {
      if (kDropout) keep_begin();
      // ---- dP = dO V^T, with the next step's keep bits behind its MFMAs; without dropout it starts at -delta
      f32x16 dp = zero16;
      if (!kDropout) {
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const f32x4 t4 = read_stat(1, g);
#pragma unroll
          for (int r = 0; r < 4; ++r) dp[4 * g + r] = t4[r];
        }
      }
      op_t xa[kRows], ob[2];
      int own_at = 0;
#pragma unroll
      for (int k = 0; k < kRows - 1; ++k) xa[k] = read_row(SM::TILE_BYTES, k);
#pragma unroll
      for (int k = 0; k < KS; ++k) {
        if (k + kRows - 1 < KS) xa[(k + kRows - 1) % kRows] = read_row(SM::TILE_BYTES, k + kRows - 1);
        if (k + 1 == KR) own_at = own_place(lane_here());
        if (k + 1 >= KR && k + 1 < KS) ob[(k + 1) & 1] = lds_read<op_t>(own_at + (k + 1 - KR) * 1024);
        dp = Tr::mfma(xa[k % kRows], k < KR ? own[k < KR ? k : 0] : ob[k & 1], dp);
        if (kDropout)
#pragma unroll
          for (int i = first_of(k, 40 - kOwn * 10, KS); i < first_of(k + 1, 40 - kOwn * 10, KS); ++i) keep_round(i);
        __builtin_amdgcn_sched_barrier(0);
      }
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");      // P is there
      // ---- dS, and dK^T += Q^T dS: the second 16 queries' dS behind the first 16's MFMAs
      const int here = lane_here(), p_at = p_place(here);
      if (kDropout) {
        lds_write(kw_place(here), word);
        keep_end();
      }
      f32x4 p4[2], d4[2];
      p4[0] = lds_read<f32x4>(p_at);
      if (kDropout) d4[0] = read_stat(1, 0);
      op_t ta[kRing];
#pragma unroll
      for (int i = 0; i < kRing - 1; ++i) ta[i] = read_tr(0, i);
      op_t sb[TS];
      float ds[2];
      auto element = [&](int E) __attribute__((always_inline)) {
        const int g = E / 4, r = E % 4;
        if (r == 0 && g < 3) {
          p4[(g + 1) & 1] = lds_read<f32x4>(p_at + (g + 1) * 1024);
          if (kDropout) d4[(g + 1) & 1] = read_stat(1, g + 1);
        }
        const float p = p4[g & 1][r];
        if (kDropout) {
          // :239-240, the sign of p says dropped; ds uses the undropped p (:242)
          int drop;
          asm("v_ashrrev_i32 %0, 31, %1" : "=v"(drop) : "v"(p));
          const int bits = __builtin_bit_cast(int, (float)dp[E]);
          ds[E & 1] = __builtin_fabsf(p) * (__builtin_bit_cast(float, __builtin_amdgcn_bitop3_b32(bits, drop, drop, 0x30)) + d4[g & 1][r]);      // (bits & ~drop)
        } else {
          ds[E & 1] = p * dp[E];
        }
        if (E & 1) {      // ds cast to Q's dtype
          const typename Tr::p2_t s2 = Tr::cvt2(ds[0], ds[1]);
          sb[E / 8][E % 8 - 1] = s2[0];
          sb[E / 8][E % 8] = s2[1];
        }
      };
      const auto rs = wave_rsrc(ds_tile, DT::BYTES);
      auto store = [&](int t) {
        const int x = lane_here(), at = ((x & 31) << 1 | x >> 5) << 4;
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_t, sb[t]), rs, at ^ (t << 7), w * 2048 + t * 1024, kDsStorePolicy);
      };
#pragma unroll
      for (int E = 0; E < 8; ++E) element(E);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < G; ++i) {
        if (i + kRing - 1 < G) ta[(i + kRing - 1) % kRing] = read_tr(0, i + kRing - 1);
        acc[i % DB] = Tr::mfma(ta[i % kRing], sb[i / DB], acc[i % DB]);
        if (i < DB)
#pragma unroll
          for (int E = 8 + first_of(i, 8, DB); E < 8 + first_of(i + 1, 8, DB); ++E) element(E);
        if (i == 0) store(0);
        if (i == DB) store(1);
        __builtin_amdgcn_sched_barrier(0);
      }
      ds_tile += DT::BYTES;
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
      next_stage();
    };
    if (kDropout) {
      keep_begin();
#pragma unroll
      for (int i = 0; i < 40 - kOwn * 10; ++i) keep_round(i);
      keep_end();
      lds_write(kw_place(lane_here()), word);
    }
    own_here();
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    for (int g = g_lo; g < g_hi; ++g) {
      const KernelArgs<BwdArgs> k = kernel_args<BwdArgs>();
      ds_tile = reinterpret_cast<char*>(k->ds_ws) + ((((int64_t)z * k->hq + hk * group + g) * k->ds_ntk + nt) * k->ds_ntq + br.lo) * DT::BYTES;
      for (int e = 0; e < ntq; ++e) step();
    }
    finish(kernel_args<BwdArgs>()->sm_scale);
  }
}

template <typename T, bool kWindowed, bool kBias, bool kDropout, int kPad>
__global__ __attribute__((amdgpu_flat_work_group_size(512, 512))) __attribute__((amdgpu_waves_per_eu(2, 2)))
void bwd_dkdv_pair_kernel(const BwdArgs a) {
  extern __shared__ __attribute__((aligned(512))) char smem_raw[];
  // one workgroup per item, in the order of bwd_dkdv_kernel
  const int xcd = blockIdx.x % kNumXcd;
  const int per_group = a.zh_group * a.num_n_tiles;
  const int parts = a.part_ws != nullptr ? a.part_heads * a.part_tiles : 1;
  const int lp = blockIdx.x / kNumXcd, li = lp / parts, gi = li / per_group, gr = li % per_group;
  const int zl = gi * a.zh_group + gr % a.zh_group, zh = xcd * a.zh_per_xcd + zl;
  if (zl >= a.zh_per_xcd || zh >= a.num_zh) return;
  int z, hk;
  split_zh(zh, a.num_zh / a.hk, 1, z, hk);
  dkdv_pair_item<T, kWindowed, kBias, kDropout, kPad>(a, hk, gr / a.zh_group, z, lp % parts, smem_raw);
}

template <typename T, int kPad, bool W, bool B, bool P>
hipError_t launch_pair_variant(const BwdArgs& a0, hipStream_t stream) {
  using SM = PairSmem<B>;
  BwdArgs a = a0;
  a.num_n_tiles = (a.seq.max_seqlen_k + SM::BN - 1) / SM::BN;
  set_work(a, tile_work(bwd_nseq(a) * a.hk, 2, a.num_n_tiles * (a.part_ws != nullptr ? a.part_heads * a.part_tiles : 1)));
  const dim3 grid((unsigned)(kNumXcd * bwd_workers(SM::D, B, a.items_per_xcd, a.num_cu, 1)));
  hipError_t e = launch_with_lds<bwd_dkdv_pair_kernel<T, W, B, P, kPad>>(grid, 512, SM::BYTES, stream, a);
  if (e == hipSuccess && a.part_ws != nullptr) e = launch_combine_dkdv<T, SM::D>(a, stream);
  return e;
}
template <typename T, int kPad>
hipError_t launch_bwd_dkdv_pair(const BwdArgs& a, bool windowed, bool bias, bool dropout, hipStream_t stream) {
#define FA_CALL(W, B, P) launch_pair_variant<T, kPad, W, B, P>(a, stream)
  FA_BWD_SWITCH(FA_CALL)
#undef FA_CALL
}

}  // namespace fa
