// Kernel argument blocks shared by the host dispatcher and the gfx950 kernels.
// Strides are in elements; the innermost stride of every tensor is 1.
#pragma once
#include <stdint.h>

namespace fa {

constexpr int kNumXcd = 8;   // MI355X: 8 XCDs x 32 CUs, one L2 each

// The 1-D work list of a kernel over the tiles of (batch element or sequence, head) pairs: each XCD owns a
// contiguous range of pairs and walks them `zh_group` at a time.  Launchers and fa_query_*_config form it here.
struct TileWork {
  int32_t num_zh, zh_per_xcd, zh_group, items_per_xcd;   // items: incl. the padding of the last group
};
inline TileWork tile_work(int num_zh, int zh_group, int items_per_pair) {
  TileWork w{num_zh, (num_zh + kNumXcd - 1) / kNumXcd, zh_group, 0};
  w.items_per_xcd = (w.zh_per_xcd + zh_group - 1) / zh_group * zh_group * items_per_pair;
  return w;
}
// pairs walked together by the kernels over q-heads (the q-heads of a GQA group share K and V)
inline int q_head_group(int hq, int hk) {
  const int ratio = hq / hk;
  return ratio > 2 ? (ratio > 8 ? 8 : ratio) : 2;
}
// persistent workgroups per XCD: `per_cu` per CU, at most one per item
inline int tile_workers(int items_per_xcd, int num_cu, int per_cu) {
  int w = num_cu / kNumXcd * per_cu;
  if (w < 1) w = 1;
  return w > items_per_xcd ? items_per_xcd : w;
}

// What the busiest worker of an XCD with the full number of pairs has to do in the persistent walk (worker_pos, one
// workgroup per CU): cost[t] is that of the t-th tile of a pair in the walk's order.
inline double walk_time(const TileWork& w, const float* cost, int tiles, int num_cu) {
  const int workers = tile_workers(w.items_per_xcd, num_cu, 1);
  double sum = 0, most = 0;
  if (workers > 64 || w.items_per_xcd > 8192) {      // one item per worker, or so many that they balance
    for (int t = 0; t < tiles; ++t) { sum += cost[t]; most = cost[t] > most ? cost[t] : most; }
    sum = sum * w.zh_per_xcd / (workers > 0 ? workers : 1);
    return sum > most ? sum : most;
  }
  double load[64] = {};
  int at = 0, step = 1;      // the worker of the next item (counted along: a division per item would show in the host's time)
  for (int first = 0; first < w.zh_per_xcd; first += w.zh_group)
    for (int t = 0; t < tiles; ++t)
      for (int i = 0; i < w.zh_group; ++i) {
        if (first + i < w.zh_per_xcd && first + i < w.num_zh) load[at] += cost[t];
        if (at + step < 0 || at + step == workers) step = -step;
        else at += step;
      }
  for (int p = 0; p < workers; ++p) most = load[p] > most ? load[p] : most;
  return most;
}

// The same with per_cu workgroups on a CU: the time of the busiest CU.  The workgroups of a CU run side by side; with l + 1 of
// them left, what remains of each takes alone[l] of what its cost says (alone[per_cu - 1] = 1: costs are those of a full CU).
// For walks of at most 64 CUs and 1024 items per XCD.
inline float walk_time_shared(const TileWork& w, const float* cost, int tiles, int num_cu, int per_cu, const float* alone) {
  const int workers = tile_workers(w.items_per_xcd, num_cu, per_cu), cus = num_cu / kNumXcd < workers ? num_cu / kNumXcd : workers;
  float of[256];      // by position in the walk's rows
  for (int q = 0; q < workers; ++q) of[q] = 0;
  int at = 0, step = 1;
  for (int first = 0; first < w.zh_per_xcd; first += w.zh_group) {
    const int heads = w.zh_per_xcd - first < w.zh_group ? w.zh_per_xcd - first : w.zh_group;
    for (int t = 0; t < tiles; ++t)
      for (int i = 0; i < w.zh_group; ++i) {
        if (i < heads) of[at] += cost[t];
        if (at + step < 0 || at + step == workers) step = -step;
        else at += step;
      }
  }
  float most = 0;
  for (int c = 0; c < cus; ++c) {
    // (worker_pos: the workgroups past the first cus sit in the row back to front)
    float l[4];
    int n = 0;
    for (int p = c; p < workers; p += cus) {
      const float x = of[p < cus ? p : cus + workers - 1 - p];
      int k = n++;
      for (; k > 0 && l[k - 1] > x; --k) l[k] = l[k - 1];
      l[k] = x;
    }
    float time = 0, before = 0;
    for (int i = 0; i < n; ++i) {
      time += (l[i] - before) * alone[n - 1 - i];
      before = l[i];
    }
    most = time > most ? time : most;
  }
  return most;
}

// Do the rows of a bias start at 16-byte boundaries, with unit column stride?
inline bool bias_aligned(const void* bias, int64_t sz, int64_t sh, int64_t sm, int64_t sn) {
  return sn == 1 && ((sz | sh | sm) & 7) == 0 && ((uintptr_t)bias & 15) == 0;
}

// Workgroups per XCD of the dK/dV and dQ kernels: one per CU (two: kTwoWaves), at most one per item.  With a
// bias the kernels get one workgroup per item instead (the loop of a workgroup then runs
// once): measured at B2 H16 S8192 D256 with window, bias, dB and dropout the persistent
// grid was 10 % slower, while it gains 1 % at the headline shape and 12 % on packed
// sequences of very different lengths.  D = 256 also gets one workgroup per item: its
// dK/dV kernel has no register to spare for the loop.
inline int bwd_workers(int head_dim, bool bias, int items_per_xcd, int num_cu, int per_cu) {
  return bias || head_dim >= 256 ? items_per_xcd : tile_workers(items_per_xcd, num_cu > 0 ? num_cu : 256, per_cu);
}

struct Strides3 {   // batch, head, row
  int64_t z, h, s;
};

struct SeqArgs {
  const int32_t* cu_q;   // null when dense
  const int32_t* cu_k;
  const int32_t* ss_q;   // strided varlen only
  const int32_t* ss_k;
  int32_t num_seqlens;   // >0 compact/strided, <0 padded, 0 dense (attn_fwd.cc:99)
  int32_t max_seqlen_q;
  int32_t max_seqlen_k;
};

struct MaskArgs {
  int32_t causal_type;   // 0 or 3
  int32_t window_left;   // raw (sentinels allowed)
  int32_t window_right;
};

struct DropoutArgs {
  float p;
  const uint64_t* seed_ptr;
  const uint64_t* offset1_ptr;
  uint64_t offset2;
};

struct FwdArgs {
  const void* q; const void* k; const void* v; const void* bias;
  void* out; float* lse;
  Strides3 sq, sk, sv, so;
  int64_t sb_z, sb_h, sb_m, sb_n;
  int32_t batch, hq, hk;
  int32_t head_dim;      // columns of Q and K (<= the compiled head dim; a multiple of 8 unless `elementwise`)
  int32_t head_dim_v;    // columns of V, Out and dOut (same bounds)
  int32_t elementwise;   // rows are not made of aligned 16-byte pieces: the vector-ALU kernels move single elements
  float sm_scale;
  SeqArgs seq;
  MaskArgs mask;
  DropoutArgs drop;
  uint64_t* seed_out; uint64_t* offset_out;
  int32_t* atomic_counter;
  int32_t num_cu;        // CUs of the device (host fills it in)
  int32_t num_m_tiles;
  int32_t num_zh;        // (batch or sequences) x q-heads
  int32_t zh_per_xcd;    // ceil(num_zh / 8)
  int32_t zh_group;      // heads walked together on one XCD
  int32_t items_per_xcd; // Q tiles (incl. padding of the last group) per XCD
  // keys split over workgroups (fa_fwd_rows.h, fwd_item's kSplit): parts, and their fp32 sums and row
  // statistics in scratch memory, laid out as combine_rows_kernel describes
  int32_t half_tiles;    // tiles of 128 rows: their workgroups per CU, 2 or (D = 64) 3; 0: whole tiles (fwd_small_tiles)
  int32_t splits;        // <= 1: not split (kernels without kSplit do not look at it); at most 64
  int32_t row_blocks;    // blocks of rows per pair
  int32_t part_rows;     // rows stored per block
  int32_t part_group, part_block;
  float* part_o;         // columns: the compiled head dim
  float* part_ml;        // reference maximum (units of the scores) and row sum
  int32_t key_mask;      // the bias is one byte per key, the same for all rows (sb_m = 0): 0 hides the key
};

struct BwdArgs {
  const void* q; const void* k; const void* v; const void* bias;
  const void* out; const void* dout;
  void* dq; void* dk; void* dv; void* db;
  const float* lse; float* delta;
  Strides3 sq, sk, sv, so, sdo, sdq, sdk, sdv;
  int64_t sb_z, sb_h, sb_m, sb_n;
  int64_t sdb_z, sdb_h, sdb_m, sdb_n;
  int32_t batch, hq, hk;
  int32_t head_dim;      // columns of Q and K (<= the compiled head dim; a multiple of 8 unless `elementwise`)
  int32_t head_dim_v;    // columns of V, Out and dOut (same bounds)
  int32_t elementwise;   // rows are not made of aligned 16-byte pieces: the vector-ALU kernels move single elements
  float sm_scale;
  SeqArgs seq;
  MaskArgs mask;
  DropoutArgs drop;
  int32_t num_m_tiles, num_n_tiles;
  int32_t num_zh;        // (batch or sequences) x heads of the launched kernel's grid
  int32_t zh_per_xcd;    // ceil(num_zh / 8)
  int32_t zh_group;      // heads walked together on one XCD
  int32_t num_cu;        // CUs of the device (host fills it in)
  int32_t items_per_xcd; // work items (incl. padding of the last group) per XCD
  int32_t walk_group;    // the wide kernels' zh_group, chosen by the host (bwd_route)
  // dS kept in HBM between the dK/dV kernel (writes it) and the dQ kernel that only does dQ = dS K:
  // tiles of 128 keys x (the dK/dV step's queries), ds_ntk x ds_ntq of them per (batch element, q-head)
  void* ds_ws;           // null: dS is not stored
  int32_t ds_ntq, ds_ntk;
  // with ds_ws: row statistics as that dK/dV kernel stages them, written by the delta kernel
  const float* lse_scaled;   // L / ln 2 (with dropout: minus log2 of its scale)
  const float* delta_prep;   // -delta (with dropout: times 1 - p)
  // dK/dV items cut into parts (few keys, many queries or q-heads): part_heads parts of the GQA group's
  // q-heads times part_tiles parts of the query tiles; each part's fp32 sums go to part_ws as
  // (sequence and kv-head, key tile, part, dK then dV, key, column), where a second kernel adds them up
  int32_t part_heads, part_tiles;
  float* part_ws;            // null: not cut
};

// Copy between a rank-4 tensor of any strides and head dim (unit last stride) and its packed
// image: contiguous (n0, n1, n2, dp) with dp the head dim rounded up to a multiple of 8, zeros in
// the excess columns.
struct RepackArgs {
  void* strided; void* packed;
  int64_t s0, s1, s2;     // element strides of the strided tensor
  int32_t n0, n1, n2;
  int32_t d, dp;          // columns of the strided tensor / of the packed one
};

struct EncodedSoftmaxArgs {
  void* r; int64_t s_z, s_h, s_m;
  int32_t batch, heads, seqlen_q, seqlen_k;
  int32_t dtype;
  DropoutArgs drop;
};

}  // namespace fa
