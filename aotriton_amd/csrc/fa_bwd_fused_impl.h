// The backward in one launch (gfx950): dK/dV items and dQ items of a head on one grid, delta recomputed in both.
// The dQ item is the split kernel's (fa_bwd_impl.h).  The dK/dV item here computes the same as the split one, whose comments
// describe it, but its tiles pass through registers on their way into LDS, because delta comes from the O and dO pieces there.
// The split item's scalars (own_scalar, kernel_args) and DropoutFold are not in it: a build with them (85 vector and 400 scalar
// registers spilled at D = 256) accessed memory outside its tensors.  The same sources built with a window show what masked_spills
// in build.py looks for, registers that the compiler moved while lanes were off; the kernel as it stands has none.
#pragma once
#include "fa_bwd_impl.h"

namespace fa {

template <typename T, int D, int NW, int BM, bool kWindowed, bool kBias, bool kDropout, int kPad>
__device__ __forceinline__ void fused_dkdv_item(const BwdArgs& a, const int hk, const int nt, const int z, char* smem_raw) {
  using Tr = Traits<T>;
  using op_t = typename Tr::op_t;
  using q4_t = typename Tr::q4_t;
  using SM = DkDvSmem<D, BM>;
  constexpr int NT = NW * 64;
  constexpr int BN = NW * 32;
  constexpr int DC = kPad ? kPad : D;            // columns computed; those past a tensor's head dim are zero
  constexpr int KS = DC / 16, MB = BM / 32, DB = DC / 32, TS = BM / 16;
  constexpr int NCH = BM * D / 8;                // 16-byte chunks per tile, per tensor
  constexpr int CH = (NCH + NT - 1) / NT;        // chunks per thread, per tensor
  constexpr int LPR = D / 8;                     // lanes that share one row

  const int tid = threadIdx.x;
  const int wave = tid >> 6, lane = tid & 63, c = lane & 31, hi = lane >> 5;
  // columns of Q/K/dQ/dK and of V/Out/dOut/dV: <= D, multiples of 8; constants unless a head dim is rounded up
  const int d_qk = kPad ? a.head_dim : D, d_v = kPad ? a.head_dim_v : D;

  const SeqInfo si = get_seq(a.seq, z);
  const int n0 = nt * BN;
  if (n0 >= si.seqlen_k) return;

  Window w{0, 0};
  if (kWindowed) w = parse_window(a.mask.causal_type, a.mask.window_left, a.mask.window_right,
                                  si.seqlen_q, si.seqlen_k);
  w.left = w.left > (1 << 30) ? (1 << 30) : (w.left < -(1 << 30) ? -(1 << 30) : w.left);
  w.right = w.right > (1 << 30) ? (1 << 30) : (w.right < -(1 << 30) ? -(1 << 30) : w.right);
  // Rows are keys here, columns are queries: key n sees query m iff n - right <= m <= n + left
  // (bwd_kernel_dk_dv.py:268-279 passes the window transposed in the same way).
  BlockRanges br = block_ranges(kWindowed, w.right, w.left, n0, si.seqlen_k, si.seqlen_q, BN, BM);

  const int group = a.hq / a.hk;

  const int key = n0 + wave * 32 + c;
  const bool key_ok = key < si.seqlen_k;
  const int key_c = key_ok ? key : si.seqlen_k - 1;
  T* dkptr = reinterpret_cast<T*>(a.dk) + (int64_t)si.batch_index * a.sdk.z + (int64_t)hk * a.sdk.h +
             (int64_t)(si.k_start + key_c) * a.sdk.s;
  T* dvptr = reinterpret_cast<T*>(a.dv) + (int64_t)si.batch_index * a.sdv.z + (int64_t)hk * a.sdv.h +
             (int64_t)(si.k_start + key_c) * a.sdv.s;

  if (br.lo > br.hi) {   // no query sees these keys
    if (key_ok) {
      q4_t zero4 = {0, 0, 0, 0};
#pragma unroll
      for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          if (32 * db + 8 * g + 4 * hi < d_qk) *reinterpret_cast<q4_t*>(dkptr + 32 * db + 8 * g + 4 * hi) = zero4;
          if (32 * db + 8 * g + 4 * hi < d_v) *reinterpret_cast<q4_t*>(dvptr + 32 * db + 8 * g + 4 * hi) = zero4;
        }
    }
    return;
  }

  // Queries that see this lane's key form one range [q_lo, q_lo + q_rng] (none: q_none): a masked
  // tile then tests an element with one unsigned comparison (fwd_kernel_inner.py:140-160 states the
  // predicate per element: key <= m + right, key >= m - left, both inside their sequences).
  int q_lo = 0, q_hi = si.seqlen_q - 1;
  if (kWindowed) {
    q_lo = key - w.right > 0 ? key - w.right : 0;
    q_hi = key + w.left < q_hi ? key + w.left : q_hi;
  }
  const bool q_none = !key_ok || q_hi < q_lo;
  const unsigned q_rng = q_none ? 0u : (unsigned)(q_hi - q_lo);

  // K and V rows of this lane's key as B operands (k = head dim)
  const T* kptr = reinterpret_cast<const T*>(a.k) + (int64_t)si.batch_index * a.sk.z + (int64_t)hk * a.sk.h +
                  (int64_t)(si.k_start + key_c) * a.sk.s;
  const T* vptr = reinterpret_cast<const T*>(a.v) + (int64_t)si.batch_index * a.sv.z + (int64_t)hk * a.sv.h +
                  (int64_t)(si.k_start + key_c) * a.sv.s;
  constexpr bool kVLds = SM::V_BYTES > 0;       // V operands come from LDS instead of registers
  op_t kreg[KS], vreg[kVLds ? 1 : KS];
#pragma unroll
  for (int k = 0; k < KS; ++k) {
    // columns past the tensors' head dim are zero (head dims are rounded up to D)
    const op_t zero8 = {0, 0, 0, 0, 0, 0, 0, 0};
    kreg[k] = 16 * k + 8 * hi < d_qk ? *reinterpret_cast<const op_t*>(kptr + 16 * k + 8 * hi) : zero8;
    if (!kVLds) vreg[k] = 16 * k + 8 * hi < d_v ? *reinterpret_cast<const op_t*>(vptr + 16 * k + 8 * hi) : zero8;
  }

  f32x16 dk[DB], dv[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int i = 0; i < 16; ++i) { dk[db][i] = 0.f; dv[db][i] = 0.f; }

  const int ntq = br.hi - br.lo + 1;
  const int total = group * ntq;
  const float qk_scale = a.sm_scale * kLog2e;
  // lane constants of the two LDS access patterns
  const int row_a = Swz<D>::row_base(lane), tr_a0 = Swz<D>::tr_base(lane, 0), tr_a1 = Swz<D>::tr_base(lane, 1);

  auto stage_ptr = [&](int stage) { return smem_raw + stage * SM::STAGE_BYTES; };

  op_t sb[TS];                         // dS operands of the dK GEMM

  // ---- staging -----------------------------------------------------------------
  // Q and dO tiles travel global -> registers -> LDS in 16-byte pieces.  The pieces
  // are issued between the MFMAs of the running tile (loads behind S = Q K^T, LDS
  // writes behind dK^T += Q^T dS), so staging costs no issue time of its own.
  // Buffer loads with a descriptor rebased on every tile: rows past the end of the
  // sequence read as zero, and a descriptor of zero records turns the fetch after
  // the last tile into a no-op.
  static_assert(NCH % NT == 0, "threads must cover the tile evenly");
  constexpr int RPI = NT / LPR;                  // rows between two pieces of one thread
  // (The split kernel's pieces go straight into LDS; here delta is computed from the O and dO registers.)
  op_t qch[CH], doch[CH], och[CH];
  float l_stage = 0.f;
  const int r0 = tid / LPR, cc0 = tid % LPR;
  const int q_voff = cc0 * 8 < d_qk ? r0 * (int)a.sq.s * 2 + cc0 * 16 : kVoffOutOfRange,       // bytes inside a tile
            do_voff = cc0 * 8 < d_v ? r0 * (int)a.sdo.s * 2 + cc0 * 16 : kVoffOutOfRange,
            o_voff = cc0 * 8 < d_v ? r0 * (int)a.so.s * 2 + cc0 * 16 : kVoffOutOfRange;
  const int q_soff = RPI * (int)a.sq.s * 2, do_soff = RPI * (int)a.sdo.s * 2, o_soff = RPI * (int)a.so.s * 2;
  int lds_off[CH];                                                        // bytes inside a tile
#pragma unroll
  for (int k = 0; k < CH; ++k) lds_off[k] = Swz<D>::addr(r0 + k * RPI, cc0);

  // Tile base pointers advance incrementally (one 64-bit add per tensor and tile);
  // with one wave per SIMD a chain of scalar multiplies per tile is not hidden.
  const int64_t q_tile_step = (int64_t)BM * a.sq.s, do_tile_step = (int64_t)BM * a.sdo.s,
                o_tile_step = (int64_t)BM * a.so.s;
  const T* qb = nullptr; const T* dob = nullptr; const T* ob = nullptr;
  const float* lse_b = nullptr;
  auto set_head = [&](int g) {
    const int hq = hk * group + g;
    const int64_t row0 = (int64_t)si.q_start + (int64_t)br.lo * BM;
    qb = reinterpret_cast<const T*>(a.q) + (int64_t)si.batch_index * a.sq.z + (int64_t)hq * a.sq.h + row0 * a.sq.s;
    dob = reinterpret_cast<const T*>(a.dout) + (int64_t)si.batch_index * a.sdo.z + (int64_t)hq * a.sdo.h +
          row0 * a.sdo.s;
    ob = reinterpret_cast<const T*>(a.out) + (int64_t)si.batch_index * a.so.z + (int64_t)hq * a.so.h +
         row0 * a.so.s;
    lse_b = a.lse + lse_offset(si, hq, a.hq) + (int64_t)br.lo * BM;
  };
  __amdgpu_buffer_rsrc_t q_rs, do_rs, o_rs, b_rs;
  // The bias tile (BM queries x the workgroup's 128 keys) is staged through LDS like Q
  // and dO when its layout allows 16-byte loads; otherwise elements are loaded directly.
  static_assert(BN == 128, "bias staging assumes 128 keys per workgroup");
  constexpr int CHB = kBias ? (BM * 16) / NT : 0;        // 16-byte bias pieces per thread
  const bool bias_lds = kBias && a.sb_n == 1 && ((a.sb_m | a.sb_h | a.sb_z) & 7) == 0 &&
                        (reinterpret_cast<uintptr_t>(a.bias) & 15) == 0;
  op_t bch[CHB > 0 ? CHB : 1];
  const int b_voff = (tid / 16) * (int)a.sb_m * 2 + (tid % 16) * 16;   // bytes inside a bias tile
  const int b_soff = (NT / 16) * (int)a.sb_m * 2;
  const int b_lds = (tid / 16) * SM::BIAS_STR + (tid % 16) * 16;
  const T* bb = nullptr;
  const T* bb_tile = nullptr;     // bias tile being fetched, its valid rows
  int b_rows = 0;
  const int b_cols = si.seqlen_k - n0 < BN ? si.seqlen_k - n0 : BN;      // valid keys of this item
  const bool bias_plain = bias_lds && (b_cols & 7) == 0;                 // no piece straddles the end of a row
  // (g, e) = (q-head inside the GQA group, Q tile inside the range) of the tile to fetch;
  // called for consecutive tiles only; `live` false: nothing is fetched
  auto fetch_begin = [&](bool live, int g, int e) {
    if (live && e == 0) set_head(g);
    const int m0 = (br.lo + e) * BM;
    int rows = si.seqlen_q - m0 < BM ? si.seqlen_q - m0 : BM;
    rows = live ? rows : 0;
    const bool any = rows > 0;
    if (kBias) {
      if (live && e == 0)
        bb = reinterpret_cast<const T*>(a.bias) + (int64_t)si.batch_index * a.sb_z +
             (int64_t)(hk * group + g) * a.sb_h + (int64_t)br.lo * BM * a.sb_m + (int64_t)n0 * a.sb_n;
      bb_tile = bb;
      b_rows = rows;
      b_rs = wave_rsrc(bb, any && bias_lds ? ((rows - 1) * (int)a.sb_m + b_cols) * 2 : 0);
      if (live) bb += (int64_t)BM * a.sb_m;
    }
    q_rs = wave_rsrc(qb, any ? ((rows - 1) * (int)a.sq.s + d_qk) * 2 : 0);
    do_rs = wave_rsrc(dob, any ? ((rows - 1) * (int)a.sdo.s + d_v) * 2 : 0);
    o_rs = wave_rsrc(ob, any ? ((rows - 1) * (int)a.so.s + d_v) * 2 : 0);
    if (tid < BM) {
      const bool ok = tid < rows;
      l_stage = ok ? lse_b[tid] : 0.f;
    }
    if (live) {
      qb += q_tile_step; dob += do_tile_step; lse_b += BM;
      ob += o_tile_step;
    }
  };
  constexpr int FETCH_PIECES = 2 * CH + CHB;
  auto fetch_piece = [&](int i) {        // Q pieces first, then dO (and O), then bias
    if (i >= 2 * CH) {
      const int k = i - 2 * CH;
      if (bias_plain) {
        // (the usual case behind one scalar branch: the two below test per lane)
        bch[k] = __builtin_bit_cast(op_t, __builtin_amdgcn_raw_buffer_load_b128(b_rs, b_voff, k * b_soff, 0));
      } else if (bias_lds) {
        bch[k] = __builtin_bit_cast(op_t, __builtin_amdgcn_raw_buffer_load_b128(b_rs, b_voff, k * b_soff, 0));
        // The descriptor ends at the last valid element of the tile's last row.  When that is
        // not at a 16-byte boundary the piece that straddles the end loses its valid elements
        // to the range check too (a dword that holds the last of an odd number of columns reads
        // as zero): that one piece is gathered element by element.
        const int row = tid / 16 + k * (NT / 16), col = (tid % 16) * 8;
        if ((b_cols & 7) != 0 && row == b_rows - 1 && col < b_cols && col + 8 > b_cols) {
          op_t x;
#pragma unroll
          for (int e = 0; e < 8; ++e)
            x[e] = col + e < b_cols ? bb_tile[(int64_t)row * a.sb_m + col + e] : Tr::cvt(0.f);
          bch[k] = x;
        }
      } else {
        // any other layout: the piece is gathered element by element
        const int row = tid / 16 + k * (NT / 16), col = (tid % 16) * 8;
        op_t x;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const bool ok = row < b_rows && n0 + col + e < si.seqlen_k;
          x[e] = ok ? bb_tile[(int64_t)row * a.sb_m + (int64_t)(col + e) * a.sb_n] : Tr::cvt(0.f);
        }
        bch[k] = x;
      }
    } else if (i < CH) {
      qch[i] = __builtin_bit_cast(op_t, __builtin_amdgcn_raw_buffer_load_b128(q_rs, q_voff, i * q_soff, 0));
    } else {
      const int k = i - CH;
      doch[k] = __builtin_bit_cast(op_t, __builtin_amdgcn_raw_buffer_load_b128(do_rs, do_voff, k * do_soff, 0));
      och[k] = __builtin_bit_cast(op_t, __builtin_amdgcn_raw_buffer_load_b128(o_rs, o_voff, k * o_soff, 0));
    }
  };
  constexpr int STORE_PIECES = 2 * CH + CHB;
  auto store_piece = [&](int i, int stage) {   // same order as the fetches
    char* sp = stage_ptr(stage);
    if (i >= 2 * CH)
      *reinterpret_cast<op_t*>(sp + 2 * SM::TILE_BYTES + 2 * BM * 4 + b_lds + (i - 2 * CH) * (NT / 16) * SM::BIAS_STR) =
          bch[i - 2 * CH];
    else if (i < CH) *reinterpret_cast<op_t*>(sp + lds_off[i]) = qch[i];
    else *reinterpret_cast<op_t*>(sp + SM::TILE_BYTES + lds_off[i - CH]) = doch[i - CH];
  };
  auto store_stats = [&](int stage) {
    char* sp = stage_ptr(stage);
    float* Ls = reinterpret_cast<float*>(sp + 2 * SM::TILE_BYTES);
    float* Ds = Ls + BM;
    // delta recomputed from O and dO (bwd_kernel_fuse.py:307-310); the LPR threads that share a row are consecutive
    // lanes.  Without dropout -delta is staged: it is the initial value of the dP accumulators.
#pragma unroll
    for (int k = 0; k < CH; ++k) {
      float acc = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) acc += (float)och[k][e] * (float)doch[k][e];
#pragma unroll
      for (int off = LPR / 2; off > 0; off >>= 1) acc += __shfl_xor(acc, off, 64);
      if (cc0 == 0) Ds[r0 + k * RPI] = kDropout ? acc : -acc;
    }
    if (tid < BM) Ls[tid] = l_stage * kRcpLn2;                          // bwd_inner_dk_dv.py:185-186
  };

  // seed and offset of the dropout mask: read once per item, not once per tile
  DropoutState drop0{};
  if (kDropout) drop0 = make_dropout_base(a.drop, a.seq.max_seqlen_k);

  // ---- one (q-head, Q tile) step -----------------------------------------------
  auto compute = [&](auto masked_tag, int g, int e, int stage, bool live, int g_nxt, int e_nxt) {
    constexpr bool masked = decltype(masked_tag)::value;
    constexpr int G1 = KS * MB, G4 = TS * DB;
    const int hq = hk * group + g;
    const int m0 = (br.lo + e) * BM;
    char* sp = stage_ptr(stage);
    const char* Qb = sp;
    const char* dOb = sp + SM::TILE_BYTES;
    const float* Ls = reinterpret_cast<const float*>(sp + 2 * SM::TILE_BYTES);
    const float* Ds = Ls + BM;
    // The staged bias tile is row-major (queries x keys) and a lane needs its key's column: a
    // transposing read hands each lane four consecutive queries of its key (lane i of a group of
    // 16 gets, in slot j, element i % 4 of the 8 bytes addressed by lane 4 j + i / 4).
    const char* Bt = sp + 2 * SM::TILE_BYTES + 2 * BM * 4 + (4 * hi + (lane & 15) / 4) * SM::BIAS_STR +
                     (wave * 32 + 16 * ((lane >> 4) & 1) + 4 * (lane & 3)) * 2;

    f32x16 s[MB], dp[MB];
    const f32x16 zero16 = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};

    DropoutState dst{};
    if (kDropout) dst = dropout_for_head(drop0, z, hq, a.hq, a.seq.max_seqlen_q);
    // The vector ALU work is spread over the MFMAs of the GEMMs that do not depend on
    // it: p = exp2(...) of S runs behind the MFMAs of dP, ds = p (dP - delta) behind
    // those of dV.  Fences keep the hand-made order.
    constexpr int kAhead = D >= 256 ? 1 : 2;
    op_t xa[kAhead + 1][MB];
    op_t pb[TS];
    uint32_t kw[kDropout ? MB : 1][4];
    // row statistics are read four rows at a time, one read ahead of their use
    f32x4 l4[2], d4[2];
    auto stat_ptr = [&](const float* base, int q) { return base + 32 * (q / 4) + 8 * (q % 4) + 4 * hi; };

    // ---- S = Q K^T ---------------------------------------------------------------
#pragma unroll
    for (int k = 0; k < kAhead; ++k)
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) xa[k][mb] = swz_read_row<T, D>(Qb, row_a, k, mb);
    if (!kDropout) {
      // dP starts at -delta of its query rows, so dP - delta leaves the matrix pipe; with
      // dropout the mask and the scale come between the two and the subtraction stays in ds_el
#pragma unroll
      for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const f32x4 t4 = *reinterpret_cast<const f32x4*>(stat_ptr(Ds, 4 * mb + g));
#pragma unroll
          for (int r = 0; r < 4; ++r) dp[mb][4 * g + r] = t4[r];
        }
    }
#pragma unroll
    // (the operand ring runs on from the Q rows of S into the dO rows of dP: the first dO operands are
    // requested behind the last MFMAs of S instead of in front of the first ones of dP)
    for (int k = 0; k < KS; ++k) {
#pragma unroll
      for (int mb = 0; mb < MB; ++mb)
        xa[(k + kAhead) % (kAhead + 1)][mb] = k + kAhead < KS ? swz_read_row<T, D>(Qb, row_a, k + kAhead, mb)
                                                              : swz_read_row<T, D>(dOb, row_a, k + kAhead - KS, mb);
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) {
        s[mb] = Tr::mfma(xa[k % (kAhead + 1)][mb], kreg[k], k == 0 ? zero16 : s[mb]);
        // the next tile's descriptors and global loads ride behind these MFMAs
        constexpr int every = G1 / FETCH_PIECES > 0 ? G1 / FETCH_PIECES : 1;
        const int gidx = k * MB + mb;
        if (gidx == 0) fetch_begin(live, g_nxt, e_nxt);
        if (kDropout) {
          // One Philox call yields the keep bits of 4 consecutive keys, i.e. of the 4
          // lanes of a quad, for one row: quad lane q runs the calls of the rows with
          // m % 4 == q (8 per tile of 64 rows instead of 32) and the bits are exchanged
          // with quad broadcasts when they are used.
          constexpr int calls = 4 * MB, stride = G1 / calls > 0 ? G1 / calls : 1;
          if (gidx % stride == 0 && gidx / stride < calls) {
            const int cidx = gidx / stride;
            kw[cidx / 4][cidx % 4] =
                dropout_keep4(dst, m0 + 32 * (cidx / 4) + 8 * (cidx % 4) + 4 * hi + (lane & 3), key & ~3);
          }
        }
        if (gidx % every == every - 1) {
#pragma unroll
          for (int q = 0; q < (FETCH_PIECES + G1 - 1) / G1; ++q) {
            const int piece = gidx / every * ((FETCH_PIECES + G1 - 1) / G1) + q;
            if (piece < FETCH_PIECES) fetch_piece(piece);
          }
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    // row statistics of the tile's queries and the first dO operands
    l4[0] = *reinterpret_cast<const f32x4*>(stat_ptr(Ls, 0));
    // D = 256 has no registers for the whole column: there the reads run one ahead of their use
    constexpr bool kBiasRing = D >= 256;
    typename Tr::q4_t bias4[kBias ? (kBiasRing ? 2 : 4 * MB) : 1];
    auto bias_read = [&](int q) {
      return Tr::lds_read_tr(reinterpret_cast<const T*>(Bt + (32 * (q / 4) + 8 * (q % 4)) * SM::BIAS_STR));
    };
    if (kBias) {
      if (kBiasRing) {
        bias4[0] = bias_read(0);
      } else {
#pragma unroll
        for (int q = 0; q < 4 * MB; ++q) bias4[q] = bias_read(q);
      }
    }
    const char* Vt = smem_raw + SM::V_OFF;
    op_t vl[3];          // ring of V operands when they come from LDS
    if (kVLds) {
      vl[0] = swz_read_row<T, D>(Vt, row_a, 0, wave);
      vl[1] = swz_read_row<T, D>(Vt, row_a, 1, wave);
    }

    // element E = 16*mb + i of the tile: p (kept in s, undropped) and its operand form
    const unsigned q_d = q_none ? 0x40000000u : (unsigned)(m0 + 4 * hi - q_lo);
    auto p_el = [&](int E) {
      const int mb = E / 16, i = E % 16, g = i / 4, r = i % 4;
      if (E % 4 == 0 && E + 4 < 16 * MB) l4[(E / 4 + 1) & 1] = *reinterpret_cast<const f32x4*>(stat_ptr(Ls, E / 4 + 1));
      // p = exp2(s*c + bias*log2e - L*log2e), one fma per element (bwd_inner_dk_dv.py:187-188)
      float x;
      if (kBias) {
        if (kBiasRing && E % 4 == 0 && E + 4 < 16 * MB) bias4[(E / 4 + 1) & 1] = bias_read(E / 4 + 1);
        const float bv = (float)bias4[kBiasRing ? (E / 4) & 1 : E / 4][r];
        x = __builtin_fmaf(s[mb][i], qk_scale, bv * kLog2e) - l4[(E / 4) & 1][r];
      } else {
        x = __builtin_fmaf(s[mb][i], qk_scale, -l4[(E / 4) & 1][r]);
      }
      if (masked) {
        // query m sees this lane's key iff q_lo <= m <= q_lo + q_rng; an empty range fails every element
        const bool vis = q_d + (unsigned)(32 * mb + 8 * g + r) <= q_rng;
        x = vis ? x : -__builtin_inff();
      }
      s[mb][i] = fast_exp2(x);
    };
    // keep bit of element E: held by the quad lane that ran the Philox call of its row
    auto keep_of = [&](int E) -> bool {
      const int mb = E / 16, g = (E % 16) / 4, r = E % 4;
      const int w = (int)kw[mb][g];
      int w4;
      switch (r) {       // quad_perm: [r, r, r, r]
        case 0: w4 = __builtin_amdgcn_mov_dpp(w, 0x00, 0xf, 0xf, true); break;
        case 1: w4 = __builtin_amdgcn_mov_dpp(w, 0x55, 0xf, 0xf, true); break;
        case 2: w4 = __builtin_amdgcn_mov_dpp(w, 0xaa, 0xf, 0xf, true); break;
        default: w4 = __builtin_amdgcn_mov_dpp(w, 0xff, 0xf, 0xf, true); break;
      }
      return ((uint32_t)w4 >> (lane & 3)) & 1u;
    };
    bool keep_bit[kDropout ? 16 * MB : 1];
    auto p_pair = [&](int E) {   // E odd: operand form of (E-1, E); dropout applies to the operand only
      float p0 = s[E / 16][E % 16 - 1], p1 = s[E / 16][E % 16];
      if (kDropout) {
        keep_bit[E - 1] = keep_of(E - 1);
        keep_bit[E] = keep_of(E);
        p0 = keep_bit[E - 1] ? p0 * dst.scale : 0.f;              // :200-201
        p1 = keep_bit[E] ? p1 * dst.scale : 0.f;
      }
      const typename Tr::p2_t p2 = Tr::cvt2(p0, p1);     // p cast to dO's dtype (composed_tensors.py:191-193)
      pb[E / 8][E % 8 - 1] = p2[0];
      pb[E / 8][E % 8] = p2[1];
    };
    auto ds_el = [&](int E) {
      const int mb = E / 16, i = E % 16, r = i % 4;
      if (!kDropout) {
        dp[mb][i] = s[mb][i] * dp[mb][i];                         // dp already holds dP - delta
        return;
      }
      if (E % 4 == 0 && E + 4 < 16 * MB) d4[(E / 4 + 1) & 1] = *reinterpret_cast<const f32x4*>(stat_ptr(Ds, E / 4 + 1));
      float dpv = dp[mb][i];
      dpv = keep_bit[E] ? dpv * dst.scale : 0.f;                  // :239-240
      dp[mb][i] = s[mb][i] * (dpv - d4[(E / 4) & 1][r]);          // ds uses the undropped p (:242)
    };
    auto ds_pair = [&](int E) {  // E odd: ds cast to Q's dtype
      const typename Tr::p2_t s2 = Tr::cvt2(dp[E / 16][E % 16 - 1], dp[E / 16][E % 16]);
      sb[E / 8][E % 8 - 1] = s2[0];
      sb[E / 8][E % 8] = s2[1];
    };

    // ---- dP = dO V^T, with p behind its MFMAs ------------------------------------
#pragma unroll
    for (int k = 0; k < KS; ++k) {
      if (k + kAhead < KS) {
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
          xa[(KS + k + kAhead) % (kAhead + 1)][mb] = swz_read_row<T, D>(dOb, row_a, k + kAhead, mb);
      }
      if (kVLds && k + 2 < KS) vl[(k + 2) % 3] = swz_read_row<T, D>(Vt, row_a, k + 2, wave);
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) {
        dp[mb] = Tr::mfma(xa[(KS + k) % (kAhead + 1)][mb], kVLds ? vl[k % 3] : vreg[kVLds ? 0 : k],
                          k == 0 && kDropout ? zero16 : dp[mb]);
        const int gidx = k * MB + mb;
#pragma unroll
        for (int E = first_of(gidx, 16 * MB, KS * MB); E < first_of(gidx + 1, 16 * MB, KS * MB); ++E) {
          p_el(E);
          if (E & 1) p_pair(E);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    // delta of the tile's queries, first transposed dO operands
    if (kDropout) d4[0] = *reinterpret_cast<const f32x4*>(stat_ptr(Ds, 0));
    // Transposed operands are read ahead of their MFMAs: a whole 16-query step ahead, or,
    // where that would take too many registers (D = 256), through a ring of kRing operands.
    constexpr bool kRingTa = DB >= 8;
    constexpr int kRing = 4;
    op_t ta[kRingTa ? 1 : 2][kRingTa ? kRing : DB];
    auto ta_read = [&](const char* tile, int gidx) { return swz_read_tr<T, D>(tile, tr_a0, tr_a1, gidx / DB, gidx % DB); };
    if (kRingTa) {
#pragma unroll
      for (int gi = 0; gi < kRing - 1; ++gi) ta[0][gi] = ta_read(dOb, gi);
    } else {
#pragma unroll
      for (int db = 0; db < DB; ++db) ta[0][db] = swz_read_tr<T, D>(dOb, tr_a0, tr_a1, 0, db);
    }

    // ---- dV^T += dO^T P, with ds behind its MFMAs --------------------------------
    constexpr int G3 = TS * DB;
#pragma unroll
    for (int t = 0; t < TS; ++t) {
#pragma unroll
      for (int db = 0; db < DB; ++db) {
        const int gidx = t * DB + db;
        if (kRingTa) {
          if (gidx + kRing - 1 < TS * DB) ta[0][(gidx + kRing - 1) % kRing] = ta_read(dOb, gidx + kRing - 1);
          dv[db] = Tr::mfma(ta[0][gidx % kRing], pb[t], dv[db]);
        } else {
          // (the last step requests the first Q^T operands of the dK phase: TS is even, they land in ta[0])
          ta[(t + 1) & 1 & (kRingTa ? 0 : 1)][db] = t + 1 < TS ? swz_read_tr<T, D>(dOb, tr_a0, tr_a1, t + 1, db)
                                                               : swz_read_tr<T, D>(Qb, tr_a0, tr_a1, 0, db);
          dv[db] = Tr::mfma(ta[t & 1 & (kRingTa ? 0 : 1)][db], pb[t], dv[db]);
        }
#pragma unroll
        for (int E = first_of(gidx, 16 * MB, G3); E < first_of(gidx + 1, 16 * MB, G3); ++E) {
          ds_el(E);
          if (E & 1) ds_pair(E);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    // ---- dK^T += Q^T dS ----------------------------------------------------------
    static_assert(TS % 2 == 0, "the dV phase leaves the first operands of this one in ta[0]");
    if (kRingTa) {
#pragma unroll
      for (int gi = 0; gi < kRing - 1; ++gi) ta[0][gi] = ta_read(Qb, gi);
    }
#pragma unroll
    for (int t = 0; t < TS; ++t) {
      if (!kRingTa && t + 1 < TS) {
#pragma unroll
        for (int db = 0; db < DB; ++db)
          ta[(t + 1) & 1 & (kRingTa ? 0 : 1)][db] = swz_read_tr<T, D>(Qb, tr_a0, tr_a1, t + 1, db);
      }
#pragma unroll
      for (int db = 0; db < DB; ++db) {
        if (kRingTa) {
          const int gidx = t * DB + db;
          if (gidx + kRing - 1 < TS * DB) ta[0][(gidx + kRing - 1) % kRing] = ta_read(Qb, gidx + kRing - 1);
          dk[db] = Tr::mfma(ta[0][gidx % kRing], sb[t], dk[db]);
        } else {
          dk[db] = Tr::mfma(ta[t & 1 & (kRingTa ? 0 : 1)][db], sb[t], dk[db]);
        }
        // the next tile's LDS writes ride behind these MFMAs
        constexpr int per = (STORE_PIECES + G4 - 1) / G4;
#pragma unroll
        for (int q = 0; q < per; ++q) {
          const int piece = (t * DB + db) * per + q;
          if (piece < STORE_PIECES) store_piece(piece, stage ^ 1);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    store_stats(stage ^ 1);
  };

  if (kVLds) {
    // the workgroup's V tile, rows past the sequence and columns past the head dim zero
    const T* vt = reinterpret_cast<const T*>(a.v) + (int64_t)si.batch_index * a.sv.z + (int64_t)hk * a.sv.h +
                  (int64_t)(si.k_start + n0) * a.sv.s;
    const int rows = si.seqlen_k - n0 < BN ? si.seqlen_k - n0 : BN;
    const auto v_rs = wave_rsrc(vt, ((rows - 1) * (int)a.sv.s + d_v) * 2);
    constexpr int VCH = BN * D / 8 / NT;
#pragma unroll
    for (int i = 0; i < VCH; ++i) {
      const int row = r0 + i * RPI;
      const int voff = cc0 * 8 < d_v ? row * (int)a.sv.s * 2 + cc0 * 16 : kVoffOutOfRange;
      const op_t x = __builtin_bit_cast(op_t, __builtin_amdgcn_raw_buffer_load_b128(v_rs, voff, 0, 0));
      *reinterpret_cast<op_t*>(smem_raw + SM::V_OFF + Swz<D>::addr(row, cc0)) = x;
    }
  }
  fetch_begin(true, 0, 0);
#pragma unroll
  for (int i = 0; i < FETCH_PIECES; ++i) fetch_piece(i);
#pragma unroll
  for (int i = 0; i < STORE_PIECES; ++i) store_piece(i, 0);
  store_stats(0);
  __syncthreads();
  // Per q-head the Q tiles come as [masked | full | masked]; each run has its own
  // loop so that the loop bodies are straight-line code.
  const int n_lb = br.fb_lo <= br.fb_hi ? br.fb_lo - br.lo : ntq;
  const int n_fb = br.fb_lo <= br.fb_hi ? br.fb_hi - br.fb_lo + 1 : 0;
  int it = 0;
  int g_cur = 0, e_cur = 0;
  auto step = [&](auto masked_tag) {
    const int stage = it & 1;
    int g_nxt = g_cur, e_nxt = e_cur + 1;
    if (e_nxt == ntq) { e_nxt = 0; ++g_nxt; }
    compute(masked_tag, g_cur, e_cur, stage, it + 1 < total, g_nxt, e_nxt);
    __syncthreads();
    ++it;
    g_cur = g_nxt; e_cur = e_nxt;
  };
  for (int g = 0; g < group; ++g) {
    for (int e = 0; e < n_lb; ++e) step(std::true_type{});
    for (int e = 0; e < n_fb; ++e) step(std::false_type{});
    for (int e = n_lb + n_fb; e < ntq; ++e) step(std::true_type{});
  }

  if (key_ok) {
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        q4_t k4, v4;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          k4[r] = Tr::cvt(dk[db][4 * g + r] * a.sm_scale);   // bwd_kernel_dk_dv.py:387-389
          v4[r] = Tr::cvt(dv[db][4 * g + r]);
        }
        if (32 * db + 8 * g + 4 * hi < d_qk) *reinterpret_cast<q4_t*>(dkptr + 32 * db + 8 * g + 4 * hi) = k4;
        if (32 * db + 8 * g + 4 * hi < d_v) *reinterpret_cast<q4_t*>(dvptr + 32 * db + 8 * g + 4 * hi) = v4;
      }
  }
}

// Per (batch, kv-head): num_n_tiles dK/dV items followed by num_m_tiles*(Hq/Hk) dQ items
// (modules/flash/csrc/attn_bwd_fused.cc:13-22, bwd_kernel_fuse.py:107-118), laid out on
// the same 1-D grid as the split kernels: each XCD owns a contiguous range of (batch,
// kv-head) pairs and walks them in pairs, so the tensors of the heads in flight stay in
// that XCD's L2.
template <typename T, int D, int NW, int BM, int BN, bool kWindowed, bool kBias, bool kDropout, int kPad>
__global__ __attribute__((amdgpu_flat_work_group_size(NW * 64, NW * 64)))
void bwd_fused_kernel(const BwdArgs a) {
  extern __shared__ __attribute__((aligned(16))) char smem_raw[];
  const int group = a.hq / a.hk;
  const int items = a.num_n_tiles + a.num_m_tiles * group;
  // persistent workgroups with the walk of the split kernels (one workgroup per item with a bias
  // or at D = 256, where the loop runs once)
  const int xcd = blockIdx.x % kNumXcd, p = blockIdx.x / kNumXcd, workers = gridDim.x / kNumXcd;
  const int per_group = a.zh_group * items;
  for (int r = 0; D >= 256 ? r < 1 : r * workers < a.items_per_xcd; ++r) {
    const int li = r * workers + ((r & 1) ? workers - 1 - p : p);
    if (li >= a.items_per_xcd) continue;
    const int gi = li / per_group, gr = li % per_group;
    const int zl = gi * a.zh_group + gr % a.zh_group;
    const int zh = xcd * a.zh_per_xcd + zl;
    if (zl >= a.zh_per_xcd || zh >= a.num_zh) continue;
    int z, hk;
    split_zh(zh, a.num_zh / a.hk, 1, z, hk);
    const int item = gr / a.zh_group;
    if (item < a.num_n_tiles) {
      fused_dkdv_item<T, D, NW, BM, kWindowed, kBias, kDropout, kPad>(a, hk, item, z, smem_raw);
    } else {
      const int t = item - a.num_n_tiles;
      const int h = hk * group + t / a.num_m_tiles;
      const int mt = a.num_m_tiles - 1 - t % a.num_m_tiles;
      dq_item<T, D, NW, BN, kWindowed, kBias, kDropout, true, kPad>(a, h, mt, z, smem_raw);
    }
    __syncthreads();     // the next item reuses the LDS stages
  }
}


template <typename T, int D, int kPad, bool W, bool B, bool P>
hipError_t launch_fused_variant(const BwdArgs& a0, hipStream_t stream) {
  using Tile = BwdTile<T, D, W>;
  constexpr int NW = Tile::NW, BM = kFusedBM<T, D, W>, BN = kFusedBN<T, D, W>;
  constexpr int smem = DkDvSmem<D, BM>::BYTES > DqSmem<D, BN>::BYTES ? DkDvSmem<D, BM>::BYTES : DqSmem<D, BN>::BYTES;
  BwdArgs a = a0;
  a.num_n_tiles = (a.seq.max_seqlen_k + NW * 32 - 1) / (NW * 32);
  a.num_m_tiles = (a.seq.max_seqlen_q + NW * 32 - 1) / (NW * 32);
  set_work(a, tile_work(bwd_nseq(a) * a.hk, 2, a.num_n_tiles + a.num_m_tiles * (a.hq / a.hk)));
  dim3 grid((unsigned)(kNumXcd * bwd_workers(D, B, a.items_per_xcd, a.num_cu, 1)));
  return launch_with_lds<bwd_fused_kernel<T, D, NW, BM, BN, W, B, P, kPad>>(grid, NW * 64, smem, stream, a);
}

template <typename T, int D, int kPad>
hipError_t launch_bwd_fused(const BwdArgs& a0, bool windowed, bool bias, bool dropout, hipStream_t stream) {
#define FA_CALL(W, B, P) launch_fused_variant<T, D, kPad, W, B, P>(a0, stream)
  FA_BWD_SWITCH(FA_CALL)
#undef FA_CALL
}

}  // namespace fa
