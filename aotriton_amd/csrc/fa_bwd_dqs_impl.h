// dQ from stored dS: the second half of the backward that keeps dS in HBM (gfx950, wave64,
// MFMA 32x32x16).
//
// The split backward of the reference recomputes S and dP in its dQ kernel
// (modules/flash/kernel/bwd_kernel_dq.py:45-389): 7 GEMMs for 5 of algorithmic work, the price of a
// dQ path without atomics.  With 288 GB of HBM at 8 TB/s there is a cheaper price: the dK/dV kernel,
// which forms dS = P (dP - delta) anyway, writes it out in the 16-bit type (the very operand values
// both dK and dQ are formed from), and this kernel reads it back once and only does
//   dQ^T (d x queries) += K_tile^T . dS^T      A = K^T from LDS,  B = dS^T from LDS
// i.e. 5 GEMMs in all, no atomics, one owner per dQ tile, at 2 bytes of HBM traffic each way per
// visible (query, key) pair.  The kernel is bound by that stream, not by the matrix pipe; calls with few steps by their latency.
//
// K and dS go straight into LDS, two steps ahead, counted by hand.  (Through registers, K a step and dS four steps ahead, a wait for
// K was one for every dS requested before it: memory answers in order.  us, before -> this: 1000 x 1531 D80 43 -> 39, window of 450 of 1801 keys
// B1 H8 D128 19.3 -> 17.7, B8 H12 S512 D64 with dB 26.6 -> 25.2; window of 1024, B2 H16 S8192 D256 246 -> 230.  What is slower that way: at D = 64 with dB
// where each CU has one workgroup of four steps, two of which are requested at once instead of all, 4000 x 200 17.8 -> 19.5, 4000 x 256 17.8 -> 19.5,
// B16 H16 S256 17.8 -> 18.8; D256 B2 H16 S4096 causal 181 -> 185.  Four stages: 4000 x 256 17.9, B16 H16 S256 17.7, D256 189, but 1-4 % more for other calls
// with dB; two stages: 1-2 % slower.)
//
// Keys per step at 128 columns: 64 with dB and where there are fewer workgroups than CUs, else 32.  A step has a barrier and a chain of LDS reads, with dB a
// turn through LDS as well, which a CU's only workgroup waits out; steps of 32 take half the LDS, so that a CU holds two workgroups.  us, 32 / 64 keys: with dB
// B2 H8 200 x 4000 113 / 91-95 (D80 108 / 87-88), B1 H8 S4096 causal 155 / 134, B2 H16 S2048 causal 102 / 86, B8 H16 S1024 119 / 108, B16 H16 S256 22.9 / 21.7; without,
// dropout: B1 H8 64 x 2000 26.8 / 22.0, B2 H8 200 x 4000 69 / 58.7, B1 H16 S2048 D80 causal 34.3 / 31.1, B3 H16 1000 x 1531 39.5 / 36.7; from a workgroup per CU
// on B64 H16 S128 D96 26.9 / 28.1, B32 H16 S128 17.2 / 18.0, B4 H16 1000 x 1531 43-54 / 43-57, B5 H16 with a bias 74-79 / 78-82.
//
// Layout of the stored tiles (written by dkdv_item, kStoreDs): one tile per (batch element, q-head,
// key tile of 128, query tile of BM = the dK/dV kernel's step) holds 128 x BM values as
// [key block of 32][16-query step t][64 pieces of 16 bytes].  A piece is what one lane of the dK/dV
// kernel holds as the MFMA operand of step t: its key c (lane % 32) against the queries
// 16 t + 4 hi + {0..3} and 16 t + 8 + 4 hi + {0..3} (hi = lane / 32).  It sits at piece position
// ((2 c + hi) ^ 8 (t & 1)), which is where the transposing LDS reads of this kernel want it: a wave
// copies 1 KB of a tile to LDS as it lies and reads bank-conflict free.
#pragma once
#include "fa_bwd_impl.h"
#include "fa_wide.h"

namespace fa {

template <int D, int BN>      // BN: keys per step
struct DqsSmem {     // stages of a step's K (swizzled) and of a dS area per wave
  static constexpr int NW = 8;
  static constexpr int STAGES = 3;
  static constexpr int K_BYTES = BN * D * 2;
  static constexpr int DS_WAVE = BN * 32 * 2;
  static constexpr int DS_OFF = STAGES * K_BYTES, DS_STAGE = NW * DS_WAVE;
  static constexpr int BYTES = DS_OFF + STAGES * DS_STAGE;
  static_assert(BYTES <= 160 * 1024, "LDS of a CU");
};

// One Q tile of 256 rows (8 waves x 32 queries) of head h against the key tiles that see it.
// kDb: the stored dS is also what dB is, in another layout: the wave's operands of a step go through its LDS
// area once more, into rows, and leave as 16-byte pieces (dB has unit column stride; its rows may start anywhere);
// where no stored tile is, dB is zero.  The kernel stays bound by its streams, two written or
// read once instead of one (B8 H12 S512 D64: 25 us for 50 MB in and 50 MB out, with 5 us for the statistics, where
// the dQ kernel that recomputes S and dP and writes dB took 48).
template <typename T, int D, int BN, int kPad, bool kDb>
__device__ __forceinline__ void dqs_item(const BwdArgs& a, const int h, const int mt, const int z, char* smem_raw) {
  using Tr = Traits<T>;
  using op_t = typename Tr::op_t;
  using q4_t = typename Tr::q4_t;
  using SM = DqsSmem<D, BN>;
  constexpr int S = SM::STAGES;
  using DT = DsTile<T, D>;
  constexpr int NW = SM::NW, NT = NW * 64, BM = NW * 32;
  constexpr int DB = (kPad ? kPad : D) / 32;
  constexpr int SPT = DT::BN / BN;          // steps per stored tile
  constexpr int KWS = BN / 32;              // 32-key blocks per step
  constexpr int NCK = KWS * 2;              // 1 KB pieces of dS per wave and step
  constexpr int LPR = D / 8;                // 16-byte pieces per K row
  constexpr int RPI = NT / LPR;             // rows between two pieces of one thread
  constexpr int CH = (BN * LPR) / NT;       // K pieces per thread and step
  static_assert((BN * LPR) % NT == 0 && CH >= 1, "threads must cover the K tile evenly");

  const int tid = threadIdx.x;
  const int wave_u = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63, c = lane & 31, hi = lane >> 5;
  const int d_qk = kPad ? a.head_dim : D;

  const SeqInfo si = get_seq(a.seq, z);
  const int q0 = mt * BM;
  if (q0 >= si.seqlen_q) return;

  const bool windowed = a.mask.causal_type != 0;
  Window w{0, 0};
  if (windowed) w = parse_window(a.mask.causal_type, a.mask.window_left, a.mask.window_right, si.seqlen_q, si.seqlen_k);
  w.left = w.left > (1 << 30) ? (1 << 30) : (w.left < -(1 << 30) ? -(1 << 30) : w.left);
  w.right = w.right > (1 << 30) ? (1 << 30) : (w.right < -(1 << 30) ? -(1 << 30) : w.right);
  // key tiles (of 128) that hold a key visible to some row of the workgroup
  const BlockRanges br = block_ranges(windowed, w.left, w.right, q0, si.seqlen_q, si.seqlen_k, BM, DT::BN);
  // The wave's rows lie in one stored query tile.  The dK/dV item of key tile nt visits that query
  // tile iff the tile pair holds a visible element; seen from the query tile that is the same range
  // arithmetic with rows and columns exchanged, so this range names exactly the tiles that were written.
  const int qblock = (q0 >> 5) + wave_u;                 // 32-row block of the sequence
  const int pm = qblock / (DT::BM / 32), qb = qblock % (DT::BM / 32);
  const BlockRanges bw = block_ranges(windowed, w.left, w.right, pm * DT::BM, si.seqlen_q, si.seqlen_k, DT::BM, DT::BN);

  const int hk = h / (a.hq / a.hk);
  const int row = q0 + wave_u * 32 + c;
  const bool row_ok = row < si.seqlen_q;
  const int row_c = row_ok ? row : si.seqlen_q - 1;
  T* dqptr = reinterpret_cast<T*>(a.dq) + (int64_t)si.batch_index * a.sdq.z + (int64_t)h * a.sdq.h +
             (int64_t)(si.q_start + row_c) * a.sdq.s;

  constexpr int BCR = BN / 8, BRI = 64 / BCR;      // dB: pieces per row of a step, rows per access
  T* const db_head = kDb ? reinterpret_cast<T*>(a.db) + (int64_t)si.batch_index * a.sdb_z + (int64_t)h * a.sdb_h : nullptr;
  auto db_piece = [&](int j, int i, const op_t x) {
    const int m = q0 + wave_u * 32 + BRI * i + lane / BCR, n = j * BN + lane % BCR * 8;
    if (m >= si.seqlen_q || n >= si.seqlen_k) return;
    T* p = db_head + (int64_t)m * a.sdb_m + n;
    if (n + 8 <= si.seqlen_k) {
      __builtin_memcpy(p, &x, 16);      // (rows may start anywhere)
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (n + e < si.seqlen_k) p[e] = x[e];
    }
  };
  const int j_steps = (si.seqlen_k + BN - 1) / BN;
  int db_lo = 0, db_hi = -1;      // steps whose dB comes from stored tiles

  f32x16 dq[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int i = 0; i < 16; ++i) dq[db][i] = 0.f;

  if (br.lo <= br.hi) {
    // steps of BN keys; the last one holds the sequence's last key
    const int j0 = br.lo * SPT;
    int j1 = br.hi * SPT + SPT - 1;
    const int j_end = (si.seqlen_k - 1) / BN;
    j1 = j1 < j_end ? j1 : j_end;
    const int jw0 = bw.lo * SPT, jw1 = bw.lo <= bw.hi ? bw.hi * SPT + SPT - 1 : -1;
    auto active = [&](int j) { return j >= jw0 && j <= jw1 && j <= j1; };
    db_lo = jw0;
    db_hi = jw1 < j1 ? jw1 : j1;

    // ---- K and dS of a step straight into LDS, S - 1 steps ahead (asm: what is in flight is counted by hand) ----
    const T* kbase = reinterpret_cast<const T*>(a.k) + (int64_t)si.batch_index * a.sk.z + (int64_t)hk * a.sk.h +
                     (int64_t)si.k_start * a.sk.s;
    constexpr int RWI = 64 / LPR;
    static_assert(RPI % 16 == 0 && RWI * D * 2 == 1024, "the swizzle repeats with every piece, a wave's piece is consecutive");
    const int r0 = tid / LPR, gch = (tid % LPR) ^ Swz<D>::f(r0);
    const int k_row = (int)a.sk.s * 2;
    const int k_voff = gch * 8 < d_qk ? r0 * k_row + gch * 16 : kVoffOutOfRange;
    const char* ws_head = reinterpret_cast<const char*>(a.ds_ws) +
                          ((int64_t)z * a.hq + h) * a.ds_ntk * (int64_t)a.ds_ntq * DT::BYTES;
    // What is stored for keys past the sequence may be infinite or NaN (dkdv_item), and K is zero there: the lanes whose piece is of such a key, piece
    // (2 c + hi) ^ 8 (t & 1) of each KB, bring zeros.  (Masking such tiles in dK/dV instead costs 2-6 % of that kernel: us, B16 H16 300 x 131 D64 with a
    // bias 33.5 -> 35.2, B4 H16 1000 x 1531 D80 with dropout 248 -> 258, Hq 64 Hk 8 5000 x 130 D160 280 -> 296.  Asked in every step it costs this kernel
    // 2-5 %; hence a loop of their own for the last steps.)
    const int ds_voff = lane * 16 + qb * DT::QBLOCK_BYTES, ds_key[2] = {lane >> 1, (lane ^ 8) >> 1};
    const int smem0 = lds_offset(smem_raw);
    constexpr int LOADS = CH + NCK;          // per wave and step
    int f_j = j0, f_stage = 0;
    auto fetch = [&](auto may_be_last) __attribute__((always_inline)) {
      int rows = si.seqlen_k - f_j * BN;
      rows = rows < BN ? rows : BN;
      rows = f_j <= j1 ? rows : 0;
      const auto k_rs = wave_rsrc_words(kbase + (int64_t)f_j * BN * a.sk.s, rows_extent(rows, k_row, d_qk * 2));
      const int k_at = smem0 + f_stage * SM::K_BYTES + wave_u * 1024;
      if constexpr (CH == 1) load_to_lds1(k_rs, k_voff, k_at);
      else load_to_lds(k_rs, k_voff, 0, k_at, k_voff, RPI * k_row, k_at + RPI * D * 2);
      // a wave that has nothing to fetch at this step reads through an empty descriptor: zeros, no traffic
      const int nt = f_j / SPT, from = f_j % SPT * KWS * 2048;
      const auto rs = wave_rsrc_words(ws_head + ((int64_t)nt * a.ds_ntq + pm) * DT::BYTES, active(f_j) ? DT::BYTES : 0);
      const int ds_at = smem0 + SM::DS_OFF + f_stage * SM::DS_STAGE + wave_u * SM::DS_WAVE;
#pragma unroll
      for (int i = 0; i < NCK; i += 2) {
        const int left = si.seqlen_k - f_j * BN - i * 16;
        load_to_lds_once(rs, !may_be_last || ds_key[0] < left ? ds_voff : kVoffOutOfRange, !may_be_last || ds_key[1] < left ? ds_voff : kVoffOutOfRange,
                         from + i * 1024, ds_at + i * 1024);
      }
      ++f_j;
      f_stage = f_stage == S - 1 ? 0 : f_stage + 1;
    };
    static_assert(CH <= 2 && NCK % 2 == 0, "pieces in pairs");

    // lane constants of the transposing reads: K^T rows of the swizzled tile, dS^T of the wave's area
    const int tr_a0 = Swz<D>::tr_base(lane, 0), tr_a1 = Swz<D>::tr_base(lane, 1);
    const int g16 = (lane >> 4) & 1, il = lane & 15;
    const int ds_rd = g16 * 1024 + ((((4 * hi + (il >> 2)) * 2 + (il & 1)) ^ (g16 << 3)) << 4) + ((il >> 1) & 1) * 8;

    int stage = 0;
#pragma unroll
    for (int i = 0; i < S - 1; ++i) fetch(std::true_type{});
    auto step = [&](auto may_be_last, int j) __attribute__((always_inline)) {
      // This wave's part of the step has arrived (what was requested for later ones may be under way; stores of dB, which come between, only make the
      // wait longer) and then everybody's, and everybody has left the stage that is filled next.
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" :: "n"((S - 2) * LOADS) : "memory");
      fetch(may_be_last);
      char* const ds_area = smem_raw + SM::DS_OFF + stage * SM::DS_STAGE + wave_u * SM::DS_WAVE;
      const bool act = active(j);
      if (act) {
        const char* Kb = smem_raw + stage * SM::K_BYTES;
        op_t bs[kDb ? BN / 16 : 1];
#pragma unroll
        for (int tk = 0; tk < BN / 16; ++tk) {
          const char* p = ds_area + ds_rd + (tk >> 1) * 2048 + (tk & 1) * 512;
          const q4_t lo = Tr::lds_read_tr(reinterpret_cast<const T*>(p));
          const q4_t up = Tr::lds_read_tr(reinterpret_cast<const T*>(p + 256));
          const op_t b = __builtin_shufflevector(lo, up, 0, 1, 2, 3, 4, 5, 6, 7);
          if constexpr (kDb) bs[tk] = b;
#pragma unroll
          for (int db = 0; db < DB; ++db) dq[db] = Tr::mfma(swz_read_tr<T, D>(Kb, tr_a0, tr_a1, tk, db), b, dq[db]);
        }
        if constexpr (kDb) {
          // b holds the keys 16 tk + 4 hi + {0..3} and 16 tk + 8 + 4 hi + {0..3} of the lane's row; the pieces of a
          // row of the area are exchanged by the row's number, so that rows do not share banks
#pragma unroll
          for (int tk = 0; tk < BN / 16; ++tk) {
            char* r = ds_area + c * (BN * 2) + 8 * hi;
            *reinterpret_cast<q4_t*>(r + (((2 * tk) ^ (c % BCR)) << 4)) = __builtin_shufflevector(bs[tk], bs[tk], 0, 1, 2, 3);
            *reinterpret_cast<q4_t*>(r + (((2 * tk + 1) ^ (c % BCR)) << 4)) = __builtin_shufflevector(bs[tk], bs[tk], 4, 5, 6, 7);
          }
#pragma unroll
          for (int i = 0; i < 32 / BRI; ++i) {
            const int r = BRI * i + lane / BCR;
            db_piece(j, i, *reinterpret_cast<const op_t*>(ds_area + r * (BN * 2) + (((lane % BCR) ^ (r % BCR)) << 4)));
          }
        }
      }
      stage = stage == S - 1 ? 0 : stage + 1;
    };
    int j = j0;
#pragma nounroll
    for (; j + S - 1 < j1; ++j) step(std::false_type{}, j);
#pragma nounroll
    for (; j <= j1; ++j) step(std::true_type{}, j);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");      // (LDS belongs to the workgroup no longer than it runs)
  }

  if constexpr (kDb) {
    for (int j = 0; j < j_steps; ++j)
      if (j < db_lo || j > db_hi)
#pragma unroll
        for (int i = 0; i < 32 / BRI; ++i) db_piece(j, i, op_t{});
  }
  if (row_ok) {
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        q4_t t4;
#pragma unroll
        for (int r = 0; r < 4; ++r) t4[r] = Tr::cvt(dq[db][4 * g + r] * a.sm_scale);   // bwd_kernel_dq.py:374-376
        if (32 * db + 8 * g + 4 * hi < d_qk) *reinterpret_cast<q4_t*>(dqptr + 32 * db + 8 * g + 4 * hi) = t4;
      }
  }
}

// One workgroup per Q tile on a 1-D grid: consecutive ids go round the XCDs, an XCD takes its
// (batch, q-head) pairs two at a time, the heaviest (last) tile of a causal mask first.
template <typename T, int D, int BN, int kPad, bool kDb>
__global__ __attribute__((amdgpu_flat_work_group_size(512, 512))) __attribute__((amdgpu_waves_per_eu(2, 2)))
void bwd_dqs_kernel(const BwdArgs a) {
  extern __shared__ __attribute__((aligned(16))) char smem_raw[];
  const int xcd = blockIdx.x % kNumXcd, li = blockIdx.x / kNumXcd;
  const int per_group = a.zh_group * a.num_m_tiles;
  const int gi = li / per_group, gr = li % per_group;
  const int zl = gi * a.zh_group + gr % a.zh_group;
  const int zh = xcd * a.zh_per_xcd + zl;
  if (zl >= a.zh_per_xcd || zh >= a.num_zh) return;
  const int mt = a.num_m_tiles - 1 - gr / a.zh_group;
  int z, h;
  split_zh(zh, a.num_zh / a.hq, a.hq / a.hk, z, h);
  dqs_item<T, D, BN, kPad, kDb>(a, h, mt, z, smem_raw);
}

template <typename T, int D, int kPad>
hipError_t launch_bwd_dqs(const BwdArgs& a0, hipStream_t stream) {
  BwdArgs a = a0;
  a.num_m_tiles = (a.seq.max_seqlen_q + 255) / 256;
  set_work(a, tile_work(bwd_nseq(a) * a.hq, q_head_group(a.hq, a.hk), a.num_m_tiles));
  dim3 grid((unsigned)(kNumXcd * a.items_per_xcd));
  constexpr int BN = D >= 256 ? 32 : 64;
  if (a.db != nullptr) return launch_with_lds<bwd_dqs_kernel<T, D, BN, kPad, true>>(grid, 512, DqsSmem<D, BN>::BYTES, stream, a);
  if constexpr (D == 128)
    if ((int64_t)a.num_zh * a.num_m_tiles >= a.num_cu)
      return launch_with_lds<bwd_dqs_kernel<T, D, 32, kPad, false>>(grid, 512, DqsSmem<D, 32>::BYTES, stream, a);
  return launch_with_lds<bwd_dqs_kernel<T, D, BN, kPad, false>>(grid, 512, DqsSmem<D, BN>::BYTES, stream, a);
}

}  // namespace fa
