// Operator entry points of the C ABI: argument checks (pure host, before any HIP
// call), shape derivation, tile-table lookup, launch.  Mirrors the hand-written
// operator layer of the reference (modules/flash/csrc/attn_fwd.cc:48-149,
// attn_bwd.cc:55-160, attn_debug.cc:30-69, attn_check.cc:36-46); the generated
// dispatch / kernel-image runtime underneath it is replaced by direct launches of
// kernels linked into this library.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <initializer_list>
#include <mutex>

#include "aotriton_amd/flash.h"
#include "aotriton_amd/probe.h"
#include "fa_args.h"
#include "fa_intervals.h"
#include "fa_kernels.h"

namespace {

// AOTRITON_DEBUG_LEVEL=0..5 -> stderr (include/aotriton/_internal/log.h:56-65)
int log_level() {
  static int level = [] {
    const char* e = std::getenv("AOTRITON_DEBUG_LEVEL");
    return e ? std::atoi(e) : 0;
  }();
  return level;
}
#define FA_LOG(lvl, ...)                                  \
  do {                                                    \
    if (log_level() >= (lvl)) {                           \
      std::fprintf(stderr, "[aotriton_amd] " __VA_ARGS__); \
      std::fputc('\n', stderr);                           \
    }                                                     \
  } while (0)

constexpr int kMaxDevices = 64;
struct DeviceInfo {
  std::atomic<int> state{0};   // 0 unknown, 1 filled
  bool is_gfx950 = false;
  int num_cu = 0;
  int clock_khz = 0;
  char arch[32] = {0};
};
DeviceInfo g_devices[kMaxDevices];
std::mutex g_device_mutex;

// v3src/util.cc:65-113: arch name up to ':' and CU count, memoised per device.
const DeviceInfo* device_of_stream(hipStream_t stream) {
  int dev = 0;
  hipError_t e = hipErrorUnknown;
  if (stream != nullptr) e = hipStreamGetDevice(stream, &dev);
  if (e != hipSuccess) e = hipGetDevice(&dev);
  if (e != hipSuccess || dev < 0 || dev >= kMaxDevices) return nullptr;
  DeviceInfo& d = g_devices[dev];
  if (d.state.load(std::memory_order_acquire) == 1) return &d;
  std::lock_guard<std::mutex> lock(g_device_mutex);
  if (d.state.load(std::memory_order_relaxed) == 1) return &d;
  hipDeviceProp_t prop;
  if (hipGetDeviceProperties(&prop, dev) != hipSuccess) return nullptr;
  size_t n = 0;
  while (prop.gcnArchName[n] && prop.gcnArchName[n] != ':' && n + 1 < sizeof(d.arch)) {
    d.arch[n] = prop.gcnArchName[n];
    ++n;
  }
  d.arch[n] = 0;
  d.is_gfx950 = std::strcmp(d.arch, "gfx950") == 0;
  d.num_cu = prop.multiProcessorCount > 0 ? prop.multiProcessorCount : 40;
  d.clock_khz = prop.clockRate;
  d.state.store(1, std::memory_order_release);
  return &d;
}

int device_index(const DeviceInfo* d) { return (int)(d - g_devices); }

// Delta buffer of fa_attn_bwd_noalloc: device memory that belongs to the library, one copy
// per GPU the library runs on, held until the process ends.  In host code the array's name
// is only a handle for hipGetSymbolAddress; the address the kernels get is looked up once
// per device (with that device current) and kept in g_scratch_ptr.
constexpr int64_t kScratchFloats = FA_NOALLOC_MAX_ROWS;
__device__ __align__(256) static float scratch[kScratchFloats];
float* g_scratch_ptr[kMaxDevices] = {};
std::mutex g_scratch_mutex;

hipError_t scratch_of_device(int dev, float** out) {
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (g_scratch_ptr[dev] == nullptr) {
    int cur = -1;
    hipError_t e = hipGetDevice(&cur);
    if (e != hipSuccess) return e;
    if (cur != dev && (e = hipSetDevice(dev)) != hipSuccess) return e;
    void* ptr = nullptr;
    e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (cur != dev) (void)hipSetDevice(cur);
    if (e != hipSuccess) return e;
    if (ptr == nullptr) return hipErrorInvalidSymbol;
    g_scratch_ptr[dev] = static_cast<float*>(ptr);
  }
  *out = g_scratch_ptr[dev];
  return hipSuccess;
}

// Workspace (dS of the backward that keeps it in HBM between its kernels, parts of dK/dV items, the parts of a split forward
// without an allocator, packed copies): one buffer per device
// that belongs to the library and only grows (hipMalloc once, then reused: a stream-ordered pool
// allocation made the host wait for the GPU on every call).  Calls on one device share it: the
// device's mutex covers the enqueue, and every call first waits (on the GPU) for the event recorded
// behind the last use (no work when that was on the same stream; stream handles are not compared:
// a destroyed stream's handle can come back).  The null stream is never destroyed, so uses on it
// record nothing: the next call on it is ordered already, and a call on another stream records the
// event then (recording and waiting in every call cost 4-5 us of a small backward).
// fa_trim_workspace frees the buffers.
std::atomic<int64_t> g_ws_limit{-1};        // bytes; -1: not set (environment, then default)
struct Workspace {
  void* ptr = nullptr;
  size_t bytes = 0;
  hipEvent_t done = nullptr;
  bool used = false;           // `done` stands behind the last use
  bool on_null = false;        // the last use was on the null stream and has no event yet
  std::mutex mutex;
};
Workspace g_ws[kMaxDevices];

int64_t ws_limit_bytes(int dev) {
  int64_t v = g_ws_limit.load(std::memory_order_relaxed);
  if (v >= 0) return v;
  static const int64_t from_env = [] {
    const char* e = std::getenv("AOTRITON_AMD_BWD_WORKSPACE_MB");
    return e ? (int64_t)std::atoll(e) << 20 : (int64_t)-1;
  }();
  if (from_env >= 0) return from_env;
  // default: an eighth of the device's memory (36 GB of 288)
  static std::atomic<int64_t> dflt[kMaxDevices];
  int64_t d = dflt[dev].load(std::memory_order_relaxed);
  if (d == 0) {
    hipDeviceProp_t prop;
    d = hipGetDeviceProperties(&prop, dev) == hipSuccess ? (int64_t)(prop.totalGlobalMem / 8) : ((int64_t)1 << 30);
    dflt[dev].store(d, std::memory_order_relaxed);
  }
  return d;
}

// Returns with the device's mutex held when it succeeds; ws_release drops it.
hipError_t ws_acquire(int dev, size_t need, hipStream_t stream, void** out) {
  Workspace& w = g_ws[dev];
  w.mutex.lock();
  hipError_t e = hipSuccess;
  const bool order = w.on_null && stream != nullptr;
  if (w.bytes < need || w.done == nullptr || order) {
    int cur = -1;
    e = hipGetDevice(&cur);
    if (e == hipSuccess && cur != dev) e = hipSetDevice(dev);
    if (e == hipSuccess && w.done == nullptr) e = hipEventCreateWithFlags(&w.done, hipEventDisableTiming);
    if (e == hipSuccess && w.bytes < need) {
      // (hipFree waits for the device: nothing uses the old buffer any more)
      if (w.ptr != nullptr) (void)hipFree(w.ptr);
      w.ptr = nullptr; w.bytes = 0; w.used = w.on_null = false;
      size_t grow = need + need / 8;
      e = hipMalloc(&w.ptr, grow);
      if (e != hipSuccess) {      // no room for the margin: exactly what this call needs
        (void)hipGetLastError();
        grow = need;
        e = hipMalloc(&w.ptr, grow);
      }
      if (e == hipSuccess) w.bytes = grow; else w.ptr = nullptr;
    }
    if (e == hipSuccess && order && w.on_null) {
      e = hipEventRecord(w.done, nullptr);      // behind everything on the device's null stream so far
      if (e == hipSuccess) { w.used = true; w.on_null = false; }
    }
    if (cur >= 0 && cur != dev) (void)hipSetDevice(cur);
  }
  if (e == hipSuccess && w.used) e = hipStreamWaitEvent(stream, w.done, 0);
  if (e != hipSuccess) {
    (void)hipGetLastError();
    w.mutex.unlock();
    return e;
  }
  *out = w.ptr;
  return hipSuccess;
}

void ws_release(int dev, hipStream_t stream) {
  Workspace& w = g_ws[dev];
  w.on_null = stream == nullptr;
  if (w.on_null) {
    w.used = false;
  } else if (hipEventRecord(w.done, stream) == hipSuccess) {
    w.used = true;
  } else {
    // without the event the next call cannot order itself behind this one
    (void)hipGetLastError();
    (void)hipStreamSynchronize(stream);
    w.used = false;
  }
  w.mutex.unlock();
}

// A call that holds the workspace (the repacking layer below) hands a part of it to the call it
// makes: that call must neither lock nor grow the buffer.
struct NestedWorkspace { bool active = false; void* ptr = nullptr; size_t bytes = 0; };
thread_local NestedWorkspace t_ws_nested;

bool stream_is_capturing(hipStream_t stream) {
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  return hipStreamIsCapturing(stream, &cap) != hipSuccess || cap != hipStreamCaptureStatusNone;
}

bool is_16bit(int dt) { return dt == FA_DTYPE_FLOAT16 || dt == FA_DTYPE_BFLOAT16; }

// ---- packed copies of tensors whose rows are not made of aligned 16-byte pieces ----------------
// (a head dim or a stride that is no multiple of 8 elements, a base that is not 16-byte aligned).
// The reference runs any head dim on its tuned kernels by padding it inside them
// (modules/flash/csrc/attn_fwd.cc:76-82,109, kernel/composed_tensors.py:60-93).  Here such a call
// gets contiguous copies with the head dim rounded up to a multiple of 8 (zeros in the excess
// columns, which add nothing to any dot product) in the library's workspace, runs on the MFMA
// kernels and has its results copied back; without workspace (limit, stream capture) it runs on
// the element-wise vector-ALU kernels.
int elem_bytes_of(int dt) { return dt == FA_DTYPE_FLOAT32 ? 4 : 2; }

size_t packed_bytes(const fa_tensor4& t) {
  const uint64_t dp = (t.sizes[3] + 7) / 8 * 8;
  const uint64_t n = t.sizes[0] * t.sizes[1] * t.sizes[2] * dp * (uint64_t)elem_bytes_of(t.dtype);
  return (size_t)((n + 255) & ~(uint64_t)255);
}

fa_tensor4 packed_view(const fa_tensor4& t, void* ptr) {
  fa_tensor4 v = t;
  const uint64_t dp = (t.sizes[3] + 7) / 8 * 8;
  v.ptr = (t.sizes[0] * t.sizes[1] * t.sizes[2]) != 0 ? ptr : nullptr;
  v.sizes[3] = dp;
  v.strides[3] = 1;
  v.strides[2] = dp;
  v.strides[1] = t.sizes[2] * dp;
  v.strides[0] = t.sizes[1] * t.sizes[2] * dp;
  return v;
}

hipError_t repack(const fa_tensor4& strided, const fa_tensor4& packed, bool unpack, hipStream_t stream) {
  if (packed.ptr == nullptr || strided.ptr == nullptr) return hipSuccess;
  fa::RepackArgs a{};
  a.strided = strided.ptr; a.packed = packed.ptr;
  a.s0 = (int64_t)strided.strides[0]; a.s1 = (int64_t)strided.strides[1]; a.s2 = (int64_t)strided.strides[2];
  a.n0 = (int32_t)strided.sizes[0]; a.n1 = (int32_t)strided.sizes[1]; a.n2 = (int32_t)strided.sizes[2];
  a.d = (int32_t)strided.sizes[3]; a.dp = (int32_t)packed.sizes[3];
  return fa::run_repack(elem_bytes_of(strided.dtype), unpack, a, stream);
}

// bytes of packed copies a call on the element-wise kernels would need instead
size_t fwd_copies_bytes(const fa_fwd_params* p) {
  return packed_bytes(p->Q) + packed_bytes(p->K) + packed_bytes(p->V) + packed_bytes(p->Out);
}
size_t bwd_copies_bytes(const fa_bwd_params* p) {
  size_t n = 0;
  for (const fa_tensor4* t : {&p->Q, &p->K, &p->V, &p->Out, &p->DO, &p->DQ, &p->DK, &p->DV}) n += packed_bytes(*t);
  return n;
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

constexpr int64_t kMaxRowStride = 1 << 21;   // elements; 256 rows of it stay below 2^31 bytes at 4 bytes per element

// rank-4 activation tensor: non-null unless it has no element, unit last stride.  *pieces is cleared
// when its rows are not made of aligned 16-byte pieces (a head dim or a stride that is no multiple
// of 8 elements, a base address that is not 16-byte aligned): such tensors run on the kernels that
// move single elements (the reference masks the excess columns of any head dim, attn_fwd.cc:76-82).
int check_act(const fa_tensor4& t, int dtype, bool* pieces) {
  const bool empty = (t.sizes[0] == 0 || t.sizes[1] == 0 || t.sizes[2] == 0) && t.sizes[3] > 0;
  if (t.ptr == nullptr && !empty) return FA_ERROR_INVALID_VALUE;
  if (t.dtype != dtype) return FA_ERROR_INVALID_VALUE;
  if (t.strides[3] != 1) return FA_ERROR_NOT_SUPPORTED;
  if (!aligned16(t.ptr) || t.sizes[3] % 8 != 0) *pieces = false;
  // strides travel as unsigned 64-bit numbers; one above 2^63 is a negative stride
  for (int i = 0; i < 3; ++i) {
    if (t.sizes[i] > 1 && (int64_t)t.strides[i] < 0) return FA_ERROR_NOT_SUPPORTED;
    if (t.sizes[i] > 1 && (t.strides[i] % 8) != 0) *pieces = false;
  }
  // a tile's rows are addressed with 32-bit byte offsets from the tile's first row
  if (t.sizes[2] > 1 && (int64_t)t.strides[2] > kMaxRowStride) return FA_ERROR_NOT_SUPPORTED;
  return FA_SUCCESS;
}

// L and delta: fp32, contiguous, one value per (sequence or batch element, query head, query row)
// in the layout the kernels index ((batch * Hq, max_seqlen_q) for rank-4 batches, (Hq, tokens)
// for packed sequences; modules/flash/kernel/fwd_kernel_inner.py:38-43).
int check_row_stats(const fa_tensor2& t, int64_t need) {
  if (t.dtype != FA_DTYPE_FLOAT32) return FA_ERROR_INVALID_VALUE;
  if (t.sizes[1] > 1 && t.strides[1] != 1) return FA_ERROR_NOT_SUPPORTED;
  if (t.sizes[0] > 1 && t.strides[0] != t.sizes[1]) return FA_ERROR_NOT_SUPPORTED;
  if ((int64_t)t.sizes[0] * (int64_t)t.sizes[1] < need) return FA_ERROR_INVALID_VALUE;
  return FA_SUCCESS;
}

// a contiguous fp32 (1, n) view for delta
fa_tensor2 row_stats_view(void* ptr, int64_t n) {
  fa_tensor2 t{};
  t.ptr = ptr;
  t.sizes[0] = 1; t.sizes[1] = (uint64_t)n;
  t.strides[0] = (uint64_t)n; t.strides[1] = 1;
  t.dtype = FA_DTYPE_FLOAT32;
  return t;
}

fa::Strides3 strides3(const fa_tensor4& t) {
  return fa::Strides3{(int64_t)t.strides[0], (int64_t)t.strides[1], (int64_t)t.strides[2]};
}

struct Shape {
  int batch, hq, hk, d, d_qk, d_v, max_sq, max_sk, num_seqlens;  // d: compiled head dim; d_qk, d_v: the tensors'; num_seqlens signed as in attn_fwd.cc:99
  bool windowed, bias, dropout;
  bool elementwise;       // some activation tensor is not made of aligned 16-byte pieces
  bool fused_as_split;    // backend 1 asked for where no single-launch kernel exists (fp32, head dims above 256)
  int64_t row_stats;      // elements of L and of delta
};

// Shared by forward and backward: everything that only depends on
// Q/K/V/B, the varlen descriptors and the scalar options.
int check_common(const fa_tensor4& Q, const fa_tensor4& K, const fa_tensor4& V, const fa_tensor4& B,
                 const fa_tensor1& cu_q, const fa_tensor1& cu_k, const fa_tensor1& ss_q,
                 const fa_tensor1& ss_k, int32_t max_sq, int32_t max_sk, int varlen_type,
                 int causal_type, float dropout_p, const fa_tensor0& seed, Shape* out) {
  const int dtype = Q.dtype;
  if (dtype != FA_DTYPE_FLOAT16 && dtype != FA_DTYPE_BFLOAT16 && dtype != FA_DTYPE_FLOAT32)
    return FA_ERROR_INVALID_VALUE;
  int e;
  bool pieces = true;
  if ((e = check_act(Q, dtype, &pieces)) != FA_SUCCESS) return e;
  if ((e = check_act(K, dtype, &pieces)) != FA_SUCCESS) return e;
  if ((e = check_act(V, dtype, &pieces)) != FA_SUCCESS) return e;
  Shape s{};
  s.elementwise = !pieces;
  s.batch = (int)Q.sizes[0];
  s.hq = (int)Q.sizes[1];
  s.hk = (int)K.sizes[1];
  const int dqk = (int)Q.sizes[3], dv = (int)V.sizes[3];
  if ((int)K.sizes[3] != dqk) return FA_ERROR_INVALID_VALUE;
  if (s.hk <= 0 || s.hq <= 0 || s.hq % s.hk != 0 || (int)V.sizes[1] != s.hk) return FA_ERROR_INVALID_VALUE;
  if (K.sizes[0] != Q.sizes[0] || V.sizes[0] != Q.sizes[0]) return FA_ERROR_INVALID_VALUE;
  if (K.sizes[2] != V.sizes[2]) return FA_ERROR_INVALID_VALUE;
  // Head dims are rounded up to a compiled one and the excess columns are masked in
  // the kernels (PADDED_HEAD, attn_fwd.cc:76-82,109); 16-byte granularity.  Dqk and Dv
  // may differ: both run on the compiled head dim that holds the larger one.
  if (dqk <= 0 || dqk > 512 || dv <= 0 || dv > 512) return FA_ERROR_NOT_SUPPORTED;
  s.d_qk = dqk;
  s.d_v = dv;
  const int dmax = dqk > dv ? dqk : dv;
  s.d = dmax <= 64 ? 64 : (dmax <= 128 ? 128 : (dmax <= 256 ? 256 : 512));   // 512: vector-ALU kernels
  s.max_sq = (int)Q.sizes[2];
  s.max_sk = (int)K.sizes[2];
  s.num_seqlens = 0;
  if (varlen_type < FA_VARLEN_NONE || varlen_type > FA_VARLEN_STRIDED) return FA_ERROR_INVALID_VALUE;
  if (cu_q.ptr != nullptr) {
    if (cu_k.ptr == nullptr || varlen_type == FA_VARLEN_NONE) return FA_ERROR_INVALID_VALUE;
    if (cu_q.dtype != FA_DTYPE_INT32 || cu_k.dtype != FA_DTYPE_INT32) return FA_ERROR_INVALID_VALUE;
    if (cu_q.sizes[0] < 2 || cu_k.sizes[0] != cu_q.sizes[0]) return FA_ERROR_INVALID_VALUE;
    if (max_sq <= 0 || max_sk <= 0) return FA_ERROR_INVALID_VALUE;
    const int n = (int)cu_q.sizes[0] - 1;
    s.num_seqlens = varlen_type == FA_VARLEN_PADDED ? -n : n;
    s.max_sq = max_sq;
    s.max_sk = max_sk;
    if (varlen_type == FA_VARLEN_STRIDED) {
      if (ss_q.ptr == nullptr || ss_k.ptr == nullptr) return FA_ERROR_INVALID_VALUE;
      if (ss_q.sizes[0] != cu_q.sizes[0] || ss_k.sizes[0] != cu_q.sizes[0]) return FA_ERROR_INVALID_VALUE;
    }
    if (varlen_type != FA_VARLEN_PADDED && s.batch != 1) return FA_ERROR_INVALID_VALUE;
    if (varlen_type == FA_VARLEN_PADDED && s.batch != n) return FA_ERROR_INVALID_VALUE;
  } else if (varlen_type != FA_VARLEN_NONE) {
    return FA_ERROR_INVALID_VALUE;
  }
  s.row_stats = s.num_seqlens > 0 ? (int64_t)s.hq * (int64_t)Q.sizes[2]
                                  : (int64_t)s.batch * s.hq * (int64_t)s.max_sq;
  if (causal_type != FA_CAUSAL_NONE && causal_type != FA_CAUSAL_WINDOWED) return FA_ERROR_NOT_SUPPORTED;
  s.windowed = causal_type != FA_CAUSAL_NONE;
  if (!(dropout_p >= 0.0f) || !(dropout_p < 1.0f)) return FA_ERROR_INVALID_VALUE;
  s.dropout = dropout_p > 0.0f;   // attn_fwd.cc:110
  if (s.dropout && seed.ptr == nullptr) return FA_ERROR_INVALID_VALUE;
  s.bias = B.ptr != nullptr;      // attn_fwd.cc:122
  if (s.bias) {
    if (B.dtype != dtype) return FA_ERROR_INVALID_VALUE;
    // Sequences of a varlen batch index the bias like the reference's kernels do
    // (modules/flash/kernel/fwd_kernel.py:393-395): batch stride times the batch index, which is the
    // sequence for the padded layout and 0 for packed tokens (one bias shared by all sequences), rows
    // and columns counted from the sequence's start; hence sizes (batch of Q, Hq, Max_seqlen_q, Max_seqlen_k).
    if ((int)B.sizes[0] != s.batch || (int)B.sizes[1] != s.hq || (int)B.sizes[2] != s.max_sq ||
        (int)B.sizes[3] != s.max_sk)
      return FA_ERROR_INVALID_VALUE;
    for (int i = 0; i < 4; ++i)
      if ((int64_t)B.strides[i] < 0) return FA_ERROR_NOT_SUPPORTED;
    // bias rows of a tile are addressed with 32-bit byte offsets, like the activations'
    if ((int64_t)B.strides[2] > kMaxRowStride || (int64_t)B.strides[3] > kMaxRowStride) return FA_ERROR_NOT_SUPPORTED;
  }
  *out = s;
  return FA_SUCCESS;
}

fa::SeqArgs seq_args(const Shape& s, const fa_tensor1& cu_q, const fa_tensor1& cu_k,
                     const fa_tensor1& ss_q, const fa_tensor1& ss_k, int varlen_type) {
  fa::SeqArgs r{};
  r.cu_q = static_cast<const int32_t*>(cu_q.ptr);
  r.cu_k = static_cast<const int32_t*>(cu_k.ptr);
  const bool strided = varlen_type == FA_VARLEN_STRIDED;
  r.ss_q = strided ? static_cast<const int32_t*>(ss_q.ptr) : nullptr;
  r.ss_k = strided ? static_cast<const int32_t*>(ss_k.ptr) : nullptr;
  r.num_seqlens = s.num_seqlens;
  r.max_seqlen_q = s.max_sq;
  r.max_seqlen_k = s.max_sk;
  return r;
}

void bias_args(const fa_bwd_params& p, const Shape& s, fa::BwdArgs* a) {
  a->bias = p.B.ptr;
  if (!s.bias) return;
  a->sb_z = (int64_t)p.B.strides[0]; a->sb_h = (int64_t)p.B.strides[1];
  a->sb_m = (int64_t)p.B.strides[2]; a->sb_n = (int64_t)p.B.strides[3];
}

int validate_fwd(const fa_fwd_params* p, int32_t version, const fa_options* opt, Shape* shape) {
  if (p == nullptr) return FA_ERROR_INVALID_VALUE;
  if (version != FA_FWD_PARAMS_VERSION) return FA_ERROR_INVALID_SYMBOL;   // attn_fwd.cc:53-55
  Shape s{};
  int e = check_common(p->Q, p->K, p->V, p->B, p->cu_seqlens_q, p->cu_seqlens_k, p->seq_strides_q,
                       p->seq_strides_k, p->Max_seqlen_q, p->Max_seqlen_k, p->varlen_type,
                       p->causal_type, p->dropout_p, p->philox_seed_ptr, &s);
  if (e != FA_SUCCESS) return e;
  bool pieces = !s.elementwise;
  if ((e = check_act(p->Out, p->Q.dtype, &pieces)) != FA_SUCCESS) return e;
  s.elementwise = !pieces;
  for (int i = 0; i < 4; ++i)
    if (p->Out.sizes[i] != (i == 3 ? p->V.sizes[3] : p->Q.sizes[i])) return FA_ERROR_INVALID_VALUE;
  if (p->A.ptr != nullptr) return FA_ERROR_NOT_SUPPORTED;   // alibi: USE_ALIBI=false in attn_fwd.cc:123
  if (p->L.ptr != nullptr && (e = check_row_stats(p->L, s.row_stats)) != FA_SUCCESS) return e;
  if (p->encoded_softmax.ptr != nullptr) {
    const fa_tensor4& r = p->encoded_softmax;
    if (r.strides[3] != 1) return FA_ERROR_NOT_SUPPORTED;
    if ((int)r.sizes[1] != s.hq || (int)r.sizes[2] != s.max_sq || (int)r.sizes[3] != s.max_sk)
      return FA_ERROR_INVALID_VALUE;
  }
  // a forced backend that does not exist cannot take the input (template/op.cc:57-70)
  if (opt != nullptr && opt->force_backend_index > 0) return FA_ERROR_PEER_ACCESS_UNSUPPORTED;
  if (shape) *shape = s;
  return FA_SUCCESS;
}

int bwd_backend(const fa_bwd_params* p, const fa_options* opt) {
  if (opt != nullptr && opt->force_backend_index >= 0) return opt->force_backend_index;
  if (opt != nullptr && opt->deterministic) return 0;   // attn_bwd.cc:147-148
  // without a delta buffer only the fused backend can run
  if (p->D.eager.ptr == nullptr && p->D.acquire == nullptr) return 1;
  return 0;
}

int validate_bwd(const fa_bwd_params* p, int32_t version, const fa_options* opt, Shape* shape,
                 int* backend) {
  if (p == nullptr) return FA_ERROR_INVALID_VALUE;
  if (version != FA_BWD_PARAMS_VERSION) return FA_ERROR_INVALID_SYMBOL;   // attn_bwd.cc:60-62
  Shape s{};
  int e = check_common(p->Q, p->K, p->V, p->B, p->cu_seqlens_q, p->cu_seqlens_k, p->seq_strides_q,
                       p->seq_strides_k, p->Max_seqlen_q, p->Max_seqlen_k, p->varlen_type,
                       p->causal_type, p->dropout_p, p->philox_seed_ptr, &s);
  if (e != FA_SUCCESS) return e;
  const int dt = p->Q.dtype;
  bool pieces = !s.elementwise;
  if ((e = check_act(p->Out, dt, &pieces)) != FA_SUCCESS) return e;
  if ((e = check_act(p->DO, dt, &pieces)) != FA_SUCCESS) return e;
  if ((e = check_act(p->DQ, dt, &pieces)) != FA_SUCCESS) return e;
  if ((e = check_act(p->DK, dt, &pieces)) != FA_SUCCESS) return e;
  if ((e = check_act(p->DV, dt, &pieces)) != FA_SUCCESS) return e;
  s.elementwise = !pieces;
  for (int i = 0; i < 4; ++i) {
    const auto o_i = i == 3 ? p->V.sizes[3] : p->Q.sizes[i];
    if (p->Out.sizes[i] != o_i || p->DO.sizes[i] != o_i ||
        p->DQ.sizes[i] != p->Q.sizes[i] || p->DK.sizes[i] != p->K.sizes[i] ||
        p->DV.sizes[i] != p->V.sizes[i])
      return FA_ERROR_INVALID_VALUE;
  }
  // without a query row L and delta hold nothing and may be null
  const bool no_query = p->Q.sizes[0] == 0 || p->Q.sizes[2] == 0;
  if (p->L.ptr == nullptr && !no_query) return FA_ERROR_INVALID_VALUE;
  if (p->L.ptr != nullptr && (e = check_row_stats(p->L, s.row_stats)) != FA_SUCCESS) return e;
  if (p->DB.ptr != nullptr) {
    if (!s.bias) return FA_ERROR_INVALID_VALUE;
    if (s.num_seqlens > 0) return FA_ERROR_NOT_SUPPORTED;   // packed tokens share one bias: every sequence would write the same dB rows
    if (p->DB.dtype != dt) return FA_ERROR_INVALID_VALUE;
    for (int i = 0; i < 4; ++i)
      if (p->DB.sizes[i] != p->B.sizes[i] || (int64_t)p->DB.strides[i] < 0) return FA_ERROR_INVALID_VALUE;
  }
  int be = bwd_backend(p, opt);
  if (be < 0 || be > 1) return FA_ERROR_PEER_ACCESS_UNSUPPORTED;   // e.g. the assembly backend 2
  // fp32 tensors and head dims above 256 have no single-launch kernel: backend 1 runs the split kernels
  // for them, with the caller's delta buffer when there is one and with one in the library's workspace
  // otherwise (whether the call gets that is known at launch: attn_bwd_impl)
  s.fused_as_split = be == 1 && (!is_16bit(dt) || s.d > 256);
  if (s.fused_as_split && p->D.eager.ptr != nullptr && (e = check_row_stats(p->D.eager, s.row_stats)) != FA_SUCCESS)
    return e;
  // (the fused backend on tensors whose rows are not aligned 16-byte pieces runs on packed copies; whether
  // the call gets the workspace for them is known at launch: fused_without_copies below)
  if (be == 0) {
    if (p->D.eager.ptr == nullptr && p->D.acquire == nullptr) return FA_ERROR_INVALID_VALUE;
    if (p->D.eager.ptr != nullptr && (e = check_row_stats(p->D.eager, s.row_stats)) != FA_SUCCESS) return e;
  }
  if (shape) *shape = s;
  if (backend) *backend = be;
  return FA_SUCCESS;
}

// fp32 forward at 128 columns: does it take fewer rounds of the CUs' time with 32 rows per workgroup (fa_f32_rows.hip) than
// with 64 (fa_f32.hip)?  Estimated in microseconds from measurements on an MI355X: a workgroup takes 7 us and 0.036 per key
// against 5 and 0.075, 256 of them at a time, the heaviest first, and 2 us against 0.018 per key once.  Measured, rows kernel / 64-row tiles (B H S, us): 1 16 512
// 28.5 / 50.8, 4 8 512 53.5 / 54.6, 8 8 512 105 / 98, 16 8 512 207 / 184; 4 8 1024 179 / 182, causal 116 / 167; 16 8 128
// 25.9 / 20.2, 128 8 128 182 / 112; 8 8 256 35.3 / 31.7; 64 rows of 64 keys 12.4 / 11.8, 2048 of those 158 / 74.
bool f32_fwd_rows128(const Shape& s, int64_t heads, int causal_type, int window_left, int window_right, int num_cu) {
  const int64_t tiles = heads * ((s.max_sq + 63) / 64);
  if (tiles <= 0 || s.max_sk <= 0) return true;
  if (tiles > 16 * num_cu) return false;
  auto time = [&](int rows, double once, double around, double per_key) {
    const int64_t n = (s.max_sq + rows - 1) / rows;
    double t = once;
    for (int64_t at = 0; at < heads * n; at += num_cu) {
      int64_t keys = s.max_sk;
      if (s.windowed) {
        const fa::Window w = fa::parse_window(causal_type, window_left, window_right, s.max_sq, s.max_sk);
        const fa::BlockRanges b = fa::block_ranges(true, w.left, w.right, (int)(n - 1 - at / heads) * rows, s.max_sq, s.max_sk, rows, 32);
        keys = b.hi < b.lo ? 0 : (b.hi - b.lo + 1) * 32;
      }
      t += around + per_key * (double)keys;
    }
    return t;
  };
  return time(32, 2, 7, 0.0363) < time(64, 0.018 * s.max_sk, 5, 0.075);
}

// fp32: the kernels whose waves share 32 rows (fa_f32_rows.hip) or those that split the head dim over the
// waves (fa_f32.hip)?  The first at 64 columns always (the second are compiled for 128).  At 128 columns the
// forward goes by the estimate above; the backward, whose dK/dV kernel lacks registers
// there, gains up to 128 tiles of 64 rows (4-11 %) and loses from 168 on (15-50 %).
bool f32_rows(const Shape& s, bool backward, int causal_type, int window_left, int window_right, int num_cu) {
  const int64_t nz = s.num_seqlens != 0 ? std::abs(s.num_seqlens) : s.batch;
  if (s.d == 64) return true;
  if (s.d != 128) return false;
  return backward ? nz * s.hq * ((s.max_sq + 63) / 64) <= num_cu / 2
                  : f32_fwd_rows128(s, nz * s.hq, causal_type, window_left, window_right, num_cu);
}

hipError_t run_fwd(int dtype, int d, const fa::FwdArgs& a, const Shape& s, hipStream_t stream) {
  if (s.elementwise) return fa::run_fwd_valu(dtype, d, a, stream);
  if (dtype == FA_DTYPE_FLOAT32)
    return (f32_rows(s, false, a.mask.causal_type, a.mask.window_left, a.mask.window_right, a.num_cu) ? fa::run_fwd_f32_rows : fa::run_fwd_f32)(d, a, s.windowed, s.bias, s.dropout, stream);
  if (d > 256) return fa::run_fwd_d512(dtype, a, s.windowed, s.bias, s.dropout, stream);
  const bool padded = a.head_dim != d || a.head_dim_v != d;   // head dim rounded up: the copies that mask the excess columns
  switch (d) {
    case 64: return (padded ? fa::run_fwd_d64_padded : fa::run_fwd_d64)(dtype, a, s.windowed, s.bias, s.dropout, stream);
    case 128:
      if (a.head_dim <= 96 && a.head_dim_v <= 96) return fa::run_fwd_d128_cols96(dtype, a, s.windowed, s.bias, s.dropout, stream);
      return (padded ? fa::run_fwd_d128_padded : fa::run_fwd_d128)(dtype, a, s.windowed, s.bias, s.dropout, stream);
    case 256: return (padded ? fa::run_fwd_d256_padded : fa::run_fwd_d256)(dtype, a, s.windowed, s.bias, s.dropout, stream);
  }
  return hipErrorNotSupported;
}

// How a forward is cut up: the tiles of fwd_kernel as they are, the same with the keys of a tile split
// into parts, or (rows) blocks of 32 packed rows with split keys (fa_fwd_rows.h).
struct FwdPlan {
  bool rows;
  int splits;                            // 1: nothing is split and no scratch is needed
  int row_blocks, part_rows;             // of the rows kernel
  int64_t o_bytes, bytes;                // scratch: the parts' sums, and all of it
};

// The rule compares estimated times in microseconds.  They come from measurements on one box (bf16):
// fwd_kernel takes a 256-row tile (128 at D = 256) through 64 keys in 1.2 / 1.9 / 1.9 us (D = 64 / 128 /
// 256) with all CUs busy (a quarter less on an idle chip, whose clock is higher), one workgroup per
// CU, and 6 us (7 at D = 256) around that; the rows kernel takes four waves of 32 rows through 4 x 32 keys in
// 0.9 / 1.2 / 2.6 us, two workgroups of a CU (one at D = 256) taking turns, and 4 us around that (7.2 at D = 256 for full blocks
// of rows: 32 keys, 4-9 rows 8 us, 64 rows 10.4, 256 rows 11.1); a part's sums of 256 rows cost
// 0.07 us of the whole chip's memory time at D = 128, the second launch 5 us.  Against 369 measured shapes of 1-2048
// queries and 2-10000 keys (227 are in profiles/forward_routes.txt) the estimate of whole tiles is within
// 25 % for 98 %, that of the rows kernel, which knows no HBM rate, for 79 %; the route taken is the best of
// the three, or within a tenth of it, for 98 %.  Off by more: at D = 64 256 queries of 4096 keys (split 32 us, rows 24) and 1500 causal of Hq 8
// Hk 2 (rows 32, tiles 28); at D128 B4 Hq 32 Hk 8 100 x 3000 (rows 59, split 53); at D = 256 three calls of one
// block of 27-32 rows and as many keys (rows 9.7-10.2, tiles 8.7; a test of the routes holds such calls to the rows).  The gains it decides on are larger
// (one query, 2051 keys, Hq 32 / Hk 8: 55 -> 11 us; 32 sequences of 8190 keys: 833 -> 189; 80 queries,
// 3216 keys: 88 -> 35; 1024 queries, 16384 keys: 402 -> 266).  Tiles of 128 rows (fwd_small_tiles below) are not among
// what is compared: they are asked about where this rule leaves the tiles whole.
FwdPlan fwd_plan(int dtype, const Shape& s, int causal_type, int window_left, int window_right, int num_cu) {
  FwdPlan r{};
  r.splits = 1;
  if (s.elementwise || !is_16bit(dtype) || s.d > 256 || s.dropout || s.max_sq <= 0 || s.max_sk <= 0 || s.batch <= 0) return r;
  const int64_t nz = s.num_seqlens != 0 ? std::abs(s.num_seqlens) : s.batch;
  const int group = s.hq / s.hk, bm = s.d > 128 ? 128 : 256;
  const int m_tiles = (s.max_sq + bm - 1) / bm;
  const int64_t tiles = nz * s.hq * m_tiles;
  if (tiles >= 4 * num_cu && s.max_sq >= bm) return r;      // the chip is full and so are the tiles
  const double wide = s.d / 128.0;

  // the tiles as they are or split: keys of the heaviest tile and of all of them
  int64_t most = 0, sum = 0;
  for (int mt = 0; mt < m_tiles; ++mt) {
    int64_t n = (s.max_sk + 63) / 64;
    if (s.windowed) {
      const fa::Window w = fa::parse_window(causal_type, window_left, window_right, s.max_sq, s.max_sk);
      const fa::BlockRanges b = fa::block_ranges(true, w.left, w.right, mt * bm, s.max_sq, s.max_sk, bm, 64);
      n = b.hi - b.lo + 1;
    }
    most = n > most ? n : most;
    sum += n;
  }
  const double t64 = s.d == 64 ? 1.2 : 1.9, around = s.d > 128 ? 7 : 6;
  auto tile_time = [&](int64_t parts) {
    const double rounds = (double)((tiles * parts + num_cu - 1) / num_cu);
    // tiles of about the same weight go in whole rounds, uneven ones fill each other's gaps
    const double even = (double)sum * nz * s.hq / num_cu *
                        (sum * 5 > most * m_tiles * 4 ? rounds * num_cu / (double)(tiles * parts) : 1.0);
    const double longest = (double)((most + parts - 1) / parts);
    const double busy = tiles * parts < num_cu ? (double)(tiles * parts) / num_cu : 1.0;
    return (even > longest ? even : longest) * t64 * (0.75 + 0.25 * busy) + around * rounds +
           (parts > 1 ? 5 + 0.07 * wide * tiles * parts : 0.0);
  };
  const double whole = tile_time(1);
  double best = whole;
  if (s.d <= 128 && s.num_seqlens == 0)
    for (int64_t parts = 2; parts <= 16 && parts * 2 <= most; ++parts)
      if (const double t = tile_time(parts); t < 0.9 * best) { best = t; r.splits = (int)parts; }

  const int64_t rows = (int64_t)group * s.max_sq;
  const int64_t items = (rows + 31) / 32 * nz * s.hk, blocks = (most * 64 + 31) / 32;
  int64_t splits = num_cu / items;
  const int64_t most_splits = (blocks + 3) / 4 < 64 ? (blocks + 3) / 4 : 64;
  splits = splits > most_splits ? most_splits : splits;
  splits = splits < 1 ? 1 : splits;      // (a window may hide every key)
  const double steps = (double)((blocks + 4 * splits - 1) / (4 * splits));
  const int64_t slots = (s.d > 128 ? 1 : 2) * num_cu, row_rounds = (items * splits + slots - 1) / slots;
  const double per_cu = s.d > 128 ? (double)row_rounds : (double)(items * splits) / num_cu;
  const double t128 = s.d == 64 ? 0.9 : s.d == 128 ? 1.2 : 2.6, rows_around = s.d > 128 && rows > 32 ? 7.2 : 4;
  const double rows_time = (per_cu > 1 ? per_cu : 1) * steps * t128 + rows_around * (double)row_rounds + 1 + (splits > 1 ? 4 : 0);
  // The row blocks of a (pair, part) run on one XCD (fwd_rows_kernel), so with fewer than eight of those, or a few more
  // than a multiple of eight, the busiest XCD has more than its share; with many row blocks that decides.  There the
  // blocks take the average tile's keys, and the rows kernel is refused where that is slower than whole tiles (us, whole tiles
  // / rows kernel, Hq 8 and Hk 2 unless said: 2048 queries and keys D128 57 / 157, causal 57 / 97; 1024 D256
  // 44 / 112; 1024 D64 22 / 27; 600 x 900 D256 41 / 79, Hq = Hk = 12 41 / 55; kept: 1024 D64 causal 23 / 20, Hq = Hk = 2
  // 2048 D128 55 / 32).
  const int64_t cus = num_cu >= fa::kNumXcd ? num_cu / fa::kNumXcd : 1, row_blocks = (rows + 31) / 32;
  const int64_t busiest = (nz * s.hk * splits + fa::kNumXcd - 1) / fa::kNumXcd * row_blocks;
  const int64_t busy_rounds = (busiest + slots / num_cu * cus - 1) / (slots / num_cu * cus);
  const double average = most > 0 ? (double)sum / ((double)most * m_tiles) : 1.0;
  const double load = average * (s.d > 128 ? (double)busy_rounds : (double)busiest / cus);
  const double busy_time = (load > 1 ? load : 1) * steps * t128 + rows_around * (double)busy_rounds + 1 + (splits > 1 ? 4 : 0);
  // (the lines: D = 128 and 256 level at 1.1 of these figures, D = 64, whose steps take 0.55 us on two XCDs, at 1.7)
  r.rows = rows_time < best && busy_time <= (s.d == 64 ? 1.75 : 1.08) * whole;
  int64_t stored;
  if (r.rows) {
    r.splits = (int)splits;
    r.row_blocks = (int)row_blocks;
    r.part_rows = (int)(rows < 32 ? rows : 32);
    stored = items * splits * r.part_rows;
  } else {
    stored = tiles * r.splits * bm;
  }
  r.o_bytes = stored * s.d * 4;
  r.bytes = r.o_bytes + stored * 8;
  return r;
}

// The kernel with 64 rows per wave (fa_fwd_wide.h; 16-bit types, head dims above 64 and up to 128, no bias, no dropout, a
// positive scale) for these 256-row tiles?  It takes a tile of 64 keys in 5-7 % less time and an item costs it 1.5-2.5 us
// more at its ends, where the two waves per SIMD of the other kernel cover for each other.  Measured (bf16, D128, us, other
// -> this kernel): B4 H16 S4096 causal 270 -> 255, full 485 -> 456, 1024 queries of 16384 keys Hq 32 Hk 8 262 -> 248, B4 H16 S1536
// causal 81 -> 79; left alone B16 H16 S2048 causal 291 / 299 (17 tiles an item, four rounds), S1024 full 277 / 280, B4 H16 S2048
// window 256 46 / 48.  The lines: 20 key tiles per item on average, or 10 where the items go in at most two rounds.
// Packed sequences stand for as many of their average length.
bool fwd_wide(const fa_fwd_params* p, const Shape& s, int splits, int num_cu) {
  if (s.elementwise || !is_16bit(p->Q.dtype) || s.d != 128 || s.bias || s.dropout || !(p->Sm_scale > 0.f) || s.max_sq <= 0 ||
      s.max_sk <= 0 || s.batch <= 0)
    return false;
  const int64_t nz = s.num_seqlens != 0 ? std::abs(s.num_seqlens) : s.batch;
  int sq = s.max_sq, sk = s.max_sk;
  if (s.num_seqlens != 0) {      // (the maximal lengths are the caller's word, the tensors are there)
    const int share = s.num_seqlens > 0 ? (int)nz : 1;
    sq = std::max(1, std::min(sq, (int)(p->Q.sizes[2] / share)));
    sk = std::max(1, std::min(sk, (int)(p->K.sizes[2] / share)));
  }
  const int m_tiles = (sq + 255) / 256;
  int64_t sum = 0;
  fa::Window w{0, 0};
  if (s.windowed) w = fa::parse_window(p->causal_type, p->window_left, p->window_right, sq, sk);
  for (int mt = 0; mt < m_tiles; ++mt) {
    const fa::BlockRanges b = fa::block_ranges(s.windowed, w.left, w.right, mt * 256, sq, sk, 256, 64);
    sum += b.hi - b.lo + 1;
  }
  const int64_t cus = num_cu >= fa::kNumXcd ? num_cu / fa::kNumXcd : 1;
  const int64_t rounds = ((nz * s.hq + fa::kNumXcd - 1) / fa::kNumXcd * m_tiles * splits + cus - 1) / cus;
  return sum >= (rounds <= 2 ? 10 : 20) * (int64_t)m_tiles * splits;
}

// Tiles of 128 rows, two workgroups per CU (FwdHalfTile) or at D = 64 three (FwdThirdTile), instead of 256 rows and one?
// Returns their number per CU, 0 for whole tiles (`wide`: those of the kernel with 64 rows per wave).  Per row the smaller
// tiles cost 5-20 % more; what they save is the part of the last round that whole tiles leave empty and, with a causal mask,
// the wait for the CU that got the heaviest ones.  So the walk of each is gone through, an item costing a + b * (its 64-key
// tiles), and a CU whose other workgroups are done being faster (constants fitted to 63 shapes at D = 64, each timed in all
// three ways, and 43 above: B1-32 H8-32, 64-2500 queries and keys, with and without a causal mask; us).  Against the best of
// the three the choices lose 0.9 % in the geometric mean at D = 64 (counting rounds only: 9 %, a third of the shapes more
// than 10 %) and 0.1 % above (1.7 %).  B16 H32 S325 D64 causal 40 / 33 / 29 us (256 rows / 128 twice / 128 three times), B4 H16
// S2136 D64 causal 86 / 67 / 78, B8 H32 S1369 D64 causal 114 / 152 / 134, B8 H12 S553 D128 causal 40 / 25.  Beyond eight rounds the
// whole tiles are even enough.
// A bias that differs between rows, at D = 64 without dropout: its 128-row tiles take rows at any alignment and the last,
// partial key tile in 16-byte pieces (kAnyRow), the whole tile the aligned rows of whole key tiles only, the rest element by
// element.  So the partial tile has a cost of its own per item (26 shapes, B1-16 H8-16, 64-1000 queries and keys: 0.3 % from the
// best of the three, whole tiles 49 %; B8 H12 S512 22.1 / 22.4 / 26.1 us, S520 61 / 26 / 30, S513 193 / 26 / 30, B16 H12 275 x 583
// 62 / 51 / 38); within the three rounds that this rule covers unaligned rows take no whole tiles, unless a window is bounded on the
// left.  Beyond, and with such a window, the tiles are whole (fa_query_fwd_config reports them).
// A bias with dropout: two per CU.  The 256-row tile of these kernels keeps more than fits 256 registers, so that the smaller one wins full
// rounds as well (us, 256 rows / 128 twice, window with both: D64 B1 H8 S1024 34 / 21, B2 H16 S2048 53 / 42, S8192 306 / 256; D128 40 / 26, 66 / 51,
// 407 / 338; B4 H16 S1500 98 / 51 and 109 / 61) and calls with rows for one whole tile (D64 B1 H8 64 x 64 20.0 / 8.3, B2 H16 S256 19.4 / 15.4, B64 H16
// 40 x 200 100 / 40, B4 H8 32 x 2000 130 / 75; D80 S64 11.1 / 9.2; D96 B4 H12 S128 14.1 / 12.2; D128 B1 H8 100 x 300 33 / 22, B8 H16 S256 window 29 / 19).
// Over 93 shapes of 32-3000 queries it takes 0.40-1.01 of the time.  Between the two, with 257 to 512 queries, it would as well (D64 B8 H16 S512 window
// 35 / 24, B2 H8 512 x 4000 213 / 139, D128 B16 H16 S300 84 / 53): these calls stay on the whole tiles, because the tests of those tiles (bias rows far apart
// and overlapping) are calls of that size and ask for them.
int fwd_small_tiles(const fa_fwd_params* p, const Shape& s, bool wide, int num_cu) {
  const bool key_bias = s.bias && !s.dropout && p->B.strides[2] == 0;
  const bool row_bias = s.bias && !key_bias && !s.dropout && s.d == 64 && p->B.strides[3] == 1;
  const bool drop_bias = s.bias && s.dropout && p->B.strides[3] == 1;
  const int cus = num_cu / fa::kNumXcd;
  if (s.elementwise || !is_16bit(p->Q.dtype) || s.d > 128 || (s.bias && !key_bias && !row_bias && !drop_bias) || s.num_seqlens != 0 || s.max_sq <= 0 ||
      s.max_sk <= 0 || s.batch <= 0 || cus < 1 || cus > 64)
    return 0;
  if (drop_bias) return s.max_sq <= 256 || s.max_sq > 512 ? 2 : 0;
  const int m_tiles = (s.max_sq + 255) / 256, group = fa::q_head_group(s.hq, s.hk);
  if (fa::tile_work(s.batch * s.hq, group, m_tiles).items_per_xcd > std::min((row_bias ? 3 : 8) * cus, 448)) return 0;
  fa::Window w{0, 0};
  if (s.windowed) w = fa::parse_window(p->causal_type, p->window_left, p->window_right, s.max_sq, s.max_sk);
  if (s.windowed && w.left < s.max_sq - 1) {      // bounded on the left as well: not among the fitted shapes, rounds are counted
    const int64_t heads = (s.batch * (int64_t)s.hq + fa::kNumXcd - 1) / fa::kNumXcd;
    if (row_bias) return 0;
    return (heads * m_tiles + cus - 1) / cus * 8 > (heads * ((s.max_sq + 127) / 128) + 2 * cus - 1) / (2 * cus) * 9 ? 2 : 0;
  }
  const float cols = s.d > 64 && std::max(s.d_qk, s.d_v) <= 96 ? 0.84f : 1.0f;
  const int halves = (s.max_sq + 127) / 128;
  int seen[2][1024];      // 64-key tiles of each tile of 256 and of 128 rows, in the walk's order: from the end of the sequence
  for (int i = 0; i < 2; ++i)
    for (int t = 0, bm = 256 >> i, n = i ? halves : m_tiles; t < n; ++t) {
      const fa::BlockRanges br = fa::block_ranges(s.windowed, w.left, w.right, (n - 1 - t) * bm, s.max_sq, s.max_sk, bm, 64);
      seen[i][t] = std::max(0, br.hi - br.lo + 1);
    }
  // `end`: what a key tile of `bn` keys that reaches past the last key costs on top
  auto time = [&](int per_cu, float a, float b, std::initializer_list<float> alone, float end = 0, int bn = 1) {
    float cost[1024];
    const int tiles = per_cu > 1 ? halves : m_tiles;
    const bool partial = s.max_sk % bn != 0;
    for (int t = 0; t < tiles; ++t) {
      const int n = seen[per_cu > 1][t];
      cost[t] = a + b * cols * n + (partial && n * 64 > s.max_sk / bn * bn ? end : 0.0f);
    }
    return fa::walk_time_shared(fa::tile_work(s.batch * s.hq, group, tiles), cost, tiles, num_cu, per_cu, alone.begin());
  };
  if (s.d > 64) {
    const float whole = wide ? time(1, 6.9f, 1.51f, {1}) : time(1, 6.3f, 1.74f, {1});
    return time(2, 7.3f, 1.99f, {0.78f, 1}) < 0.97f * whole ? 2 : 0;
  }
  if (row_bias) {
    const bool aligned = fa::bias_aligned(p->B.ptr, p->B.strides[0], p->B.strides[1], p->B.strides[2], p->B.strides[3]);
    const float two = time(2, 3.85f, 2.32f, {0.83f, 1}, 2.1f, 64), three = time(3, 4.54f, 3.43f, {0.72f, 0.83f, 1}, 0.85f, 32);
    if (aligned && std::min(two, three) >= 0.98f * time(1, 4.65f, 2.18f, {1}, 8.3f, 128)) return 0;
    return three < two ? 3 : 2;
  }
  const float whole = time(1, 4.35f, 1.12f, {1}), two = time(2, 4.54f, 1.27f, {0.74f, 1});
  // (with dropout three waves per SIMD have no idle vector ALU to use)
  const float three = s.dropout ? 2 * two : time(3, 5.16f, 1.93f, {0.62f, 0.78f, 1});
  return std::min(two, three) >= 0.98f * whole ? 0 : three < two ? 3 : 2;
}

hipError_t run_fwd_rows(int dtype, int d, const fa::FwdArgs& a, const Shape& s, hipStream_t stream) {
  const bool padded = a.head_dim != d || a.head_dim_v != d;
  switch (d) {
    case 64: return (padded ? fa::run_fwd_rows_d64_padded : fa::run_fwd_rows_d64)(dtype, a, s.windowed, s.bias, stream);
    case 128: return (padded ? fa::run_fwd_rows_d128_padded : fa::run_fwd_rows_d128)(dtype, a, s.windowed, s.bias, stream);
    default: return (padded ? fa::run_fwd_rows_d256_padded : fa::run_fwd_rows_d256)(dtype, a, s.windowed, s.bias, stream);
  }
}

fa::DropoutArgs dropout_args(float p, const fa_tensor0& seed, const fa_tensor0& off1, uint64_t off2) {
  fa::DropoutArgs d{};
  d.p = p;
  d.seed_ptr = static_cast<const uint64_t*>(seed.ptr);
  d.offset1_ptr = static_cast<const uint64_t*>(off1.ptr);
  d.offset2 = off2;
  return d;
}

// Bytes of workspace with which the split backward keeps dS in HBM, 0 when this call recomputes S
// and dP in its dQ kernel instead (anything but the 16-bit MFMA kernels up to 256 columns, packed sequences, an
// empty tensor, plain calls at 64 columns, and with dB what the first test below names).  *ds_bytes / *stat_bytes: the
// parts of the buffer.
int64_t ds_workspace_need(const fa_bwd_params* p, const Shape& s, int* ntq, int* ntk, int64_t* ds_bytes,
                          int64_t* stat_bytes) {
  if (s.elementwise || !is_16bit(p->Q.dtype) || (s.d != 64 && s.d != 128 && s.d != 256) || s.num_seqlens != 0 ||
      s.batch <= 0 || s.max_sq <= 0 || s.max_sk <= 0)
    return 0;
  // dB leaves the dQ-from-dS kernel as 16-byte pieces of its rows, wherever they start (rows at odd places left to the
  // recomputing one: B9 H16 S1007 D64 bf16 forward + backward 732 us, stored 576; B16 H12 S700 fp16 520 -> 383).  Columns that
  // lie apart are left to the recomputing one; so are small calls,
  // where the third launch costs what is saved (us forward + backward, recomputing -> stored: B2 H8 S256 D64
  // 50 -> 53, B8 H12 S512 D64 118 -> 100, D128 148 -> 132, D256 468 -> 420, B16 H16 S1024 D64 842 -> 795, causal 670 -> 579),
  // and long rows at D = 64.  There (us of the backward alone, recomputing -> stored, B1): H8 S4096 causal 312 -> 300, H16
  // S4096 610 -> 560, window 1000 283 -> 254, S6144 causal 793 -> 744, S8192 2195 -> 2050, window 1000 713 -> 710, but causal
  // 1272 -> 1298 and window 4000 1076 -> 1138: the line gives up 6 % of some calls for 2-6 % of others (stored tiles
  // against visible pairs would tell them apart)
  if (p->DB.ptr != nullptr &&
      ((int64_t)s.batch * s.hq * s.max_sq * s.max_sk < (int64_t)1 << 22 || (s.d == 64 && s.max_sk > 4096) ||
       p->DB.strides[3] != 1))
    return 0;
  // the 64-column build: 2 bytes per pair are too many for its little GEMM work unless the dQ kernel is
  // spared a bias or the Philox arithmetic (same box, stored / recomputing: 1.05-1.14 plain, 0.69-0.81 with either)
  if (s.d == 64 && !s.dropout && !s.bias) return 0;
  int64_t tile_bytes = 0;
  fa::ds_tile_counts(s.d, s.max_sq, s.max_sk, ntq, ntk, &tile_bytes);
  *ds_bytes = (int64_t)s.batch * s.hq * *ntq * *ntk * tile_bytes;
  *stat_bytes = (s.row_stats * 4 + 255) & ~(int64_t)255;
  return *ds_bytes + 2 * *stat_bytes;
}

// Parts of the dK/dV items (16-bit types, head dims up to 256).  An item is a 128-key tile of one kv-head
// and runs through the query tiles of all q-heads of the group, one after the other: with few kv-heads
// and short key ranges there are fewer items than CUs and each takes long.  Cut into parts (by
// q-heads first, then by query tiles) they fill the chip; the parts' fp32 sums cost a round trip and a
// launch.
struct DkdvParts { int heads, tiles; int64_t bytes; };

// The rule compares estimated times in microseconds: 1.9-2.3 per step (64 queries at D = 128, 128 at 64,
// 32 at 256; more with a bias or dropout), 7 around an item, 4 for the second launch and 0.065 of the
// chip's memory time per part (256 KB written and read at D = 128).  Head dim 64 without a bias is older than the kernel
// there, which takes 64-query steps, two workgroups per CU: the figures stand for 128 queries and one, and calls
// with more than num_cu / 2 items stay whole although there are twice as many places.  What it chooses there holds (us of
// the backward, whole / cut, B1: Hq 8 Hk 2 2048 x 256 143 / 35, Hq 16 Hk 4 1024 causal 90 / 46, H8 4096 x 512 82 / 41, H4 4096 x
// 1024 causal 88 / 50, Hq 16 Hk 8 512 x 1024 causal 36 / 34; H8 1024 x 1000 39 / 40), finer cuts have not been measured.
// `stored`: the items keep dS in HBM.
DkdvParts dkdv_parts(const fa_bwd_params* p, const Shape& s, bool stored, int num_cu) {
  DkdvParts r{1, 1, 0};
  if (s.elementwise || !is_16bit(p->Q.dtype) || s.d > 256 || s.max_sq <= 0 || s.max_sk <= 0 || s.batch <= 0) return r;
  const int64_t nz = s.num_seqlens != 0 ? std::abs(s.num_seqlens) : s.batch;
  const int n_tiles = (s.max_sk + 127) / 128, group = s.hq / s.hk;
  const int64_t items = nz * s.hk * n_tiles;
  if (items * 2 > num_cu) return r;
  const int bm = s.d == 64 ? 128 : s.d == 128 ? 64 : 32;
  int64_t most = 0, sum = 0;
  for (int nt = 0; nt < n_tiles; ++nt) {
    int64_t n = (s.max_sq + bm - 1) / bm;
    if (s.windowed) {
      const fa::Window w = fa::parse_window(p->causal_type, p->window_left, p->window_right, s.max_sq, s.max_sk);
      const fa::BlockRanges b = fa::block_ranges(true, w.right, w.left, nt * 128, s.max_sk, s.max_sq, 128, bm);
      n = b.hi - b.lo + 1;
    }
    most = n > most ? n : most;
    sum += n;
  }
  const double t_step = (s.d == 64 ? 2.3 : s.d == 128 ? 1.9 : 2.1) * (s.dropout ? 1.7 : 1.0) * (s.bias ? 1.3 : 1.0);
  // Head dim 64 with a bias and no dropout, of the cuts within some of the lowest estimate:
  // - items that store dS (kTwoDkDv): 64-query steps, two parts share a CU, and what the estimate calls level is a gain.  The lowest
  //   may be 2 % above whole items, and the finest cut within 2 % of it is taken: 16 shapes (B1-8 H1-16, 256-4096 x 128-2048), each
  //   in eight cuts, come out 1.9 % above their best in the geometric mean (the general rule: 3.6 %).  us of the backward, whole /
  //   this / the general rule: B2 H8 S1024 54.6 / 51.6 / 54.6, B1 H8 S512 34.2 / 32.8 / 34.2, B3 H2 2247 x 151 113 / 36 / 39.
  // - items that do not, as with dB in small calls: a part has a CU to itself and more of them make more rounds on the XCDs of
  //   few heads.  The coarsest cut within 8 % is taken where the lowest is below whole items: 30 shapes (B1-4 H1-24, 250-2250 x
  //   128-2000) come out 1.9 % above their best (the general rule: 3.3 %, the rule above: 3.6 %).  us, whole / this / the general rule /
  //   the rule above: B1 H2 S1400 122 / 114 / 124 / 124, S1024 82 / 66 / 66 / 76, B1 H8 S512 44.8 / 43.2 / 44.8 / 41.7.
  const bool bias64 = s.d == 64 && s.bias && !s.dropout && s.num_seqlens == 0 && p->B.strides[3] == 1;
  const bool shared = bias64 && stored && s.max_sk >= 8;
  const double whole = group * most * t_step + 7;
  double best = whole;
  auto for_cuts = [&](auto&& take) {      // from the coarsest to the finest
    for (int heads = 1; heads <= group; ++heads) {
      if (group % heads != 0) continue;
      for (int tiles = 1; tiles <= 16 && tiles <= most; ++tiles) {
        if (heads * tiles == 1 || (tiles > 1 && heads < group)) continue;
        const int64_t wgs = items * heads * tiles, rounds = (wgs + num_cu - 1) / num_cu;
        const double t = rounds * ((double)(group / heads) * ((most + tiles - 1) / tiles) * t_step + 7) + 4 +
                         0.065 * s.d / 128 * wgs;
        take(heads, tiles, t);
      }
    }
  };
  if (bias64) {
    const double level = (shared ? 1.02 : 1.0) * whole;
    best = level;
    for_cuts([&](int, int, double t) { best = std::min(best, t); });
    const double most_t = (shared ? 1.02 : 1.08) * best;
    if (best < level)
      for_cuts([&](int heads, int tiles, double t) {
        if (t <= most_t && (shared || r.heads * r.tiles == 1)) { r.heads = heads; r.tiles = tiles; }
      });
  } else {
    for_cuts([&](int heads, int tiles, double t) { if (t < 0.95 * best) { best = t; r.heads = heads; r.tiles = tiles; } });
  }
  // An XCD owns the items of its kv-heads: with fewer kv-heads than XCDs the parts may just make more rounds there.
  // Under a narrow window, whose items are alike, nothing is gained then (us of the whole backward, uncut / cut, B1 H2
  // S1536, window 200: dropout D128 49 / 67, D256 68 / 78, bias 56 / 65); items of uneven weight fill each other's gaps
  // (three packed sequences of 1500-2500 tokens, Hq 8, Hk 2, D128 causal 265 / 184).
  const int64_t cus = num_cu >= fa::kNumXcd ? num_cu / fa::kNumXcd : 1;
  const int64_t busiest = (nz * s.hk + fa::kNumXcd - 1) / fa::kNumXcd * n_tiles;
  auto xcd_time = [&](int heads, int tiles) {
    return (double)((busiest * heads * tiles + cus - 1) / cus) *
           ((double)(group / heads) * ((most + tiles - 1) / tiles) * t_step + 7);
  };
  if (s.windowed && s.num_seqlens == 0 && sum * 5 > most * n_tiles * 4 && r.heads * r.tiles > 1 &&
      xcd_time(r.heads, r.tiles) + 4 + 0.065 * s.d / 128 * items * r.heads * r.tiles > 1.05 * xcd_time(1, 1))
    r.heads = r.tiles = 1;
  if (r.heads * r.tiles > 1) r.bytes = items * r.heads * r.tiles * (2 * 128 * s.d * 4);
  return r;
}

// The kernels with 64 rows per wave (fa_bwd_wide.h; 16-bit types, head dims above 64 and up to 128, no bias, no dropout) take
// the matrix work of a pair in 8-25 % less time, in workgroups of 256 rows instead of 128: they are chosen where that does
// not leave more of the chip idle.  The rule compares the walks of both over the busiest XCD, in microseconds: an item
// takes what its steps take (128 x 64 or 256 x 32 pairs) and what it costs to begin and to end.  Fitted to 128 calls (bf16,
// D128; heads 8-512, 64-4096 tokens, causal or not, GQA, windows; us of the whole backward, 128 -> 256 rows): B16 H16 S512
// causal 136 -> 124, B8 H16 S1024 173 -> 157, B4 H16 S4096 912 -> 825, full 1584 -> 1493; left alone B8 H16 S512 causal 72 / 74,
// B1 H8 S1024 60 / 91, Hq 32 Hk 8 S2048 183 / 405.  It is off the better choice by 4 % in one of them.
// Packed sequences stand for as many of their average length, but no walk is shorter than the longest one's heaviest item.
struct BwdRoute {
  bool wide_dkdv, wide_dq;
  bool recompute;               // both, and faster than the kernels that keep dS
  int group_dkdv, group_dq;     // heads walked together by the wide kernels
};
struct WalkCost { double item, step; };
// rows: the side the items are tiles of; cols: the side they step over
double tile_walk_time(const fa_bwd_params* p, const Shape& s, bool keys, int num_heads, int zh_group, int tile, int step,
                      int heads_per_item, WalkCost c, int num_cu, int max_rows, int max_cols, int nz) {
  // Beyond kMost tiles, which any walk balances, evenly spaced ones stand for all.  (The maximal length of packed sequences is
  // the caller's word: nothing here may grow with it, neither memory nor time.)
  constexpr int kMost = 1024;
  float cost[kMost];
  const int n_tiles = (int)(((int64_t)max_rows + tile - 1) / tile), n = std::min(n_tiles, kMost);
  fa::Window w{0, 0};
  if (s.windowed)
    w = fa::parse_window(p->causal_type, p->window_left, p->window_right, keys ? max_cols : max_rows, keys ? max_rows : max_cols);
  double sum = 0, most = 0;
  for (int t = 0; t < n; ++t) {
    const int at = n == n_tiles ? t : (int)((int64_t)t * n_tiles / n);
    const fa::BlockRanges b = fa::block_ranges(s.windowed, keys ? w.right : w.left, keys ? w.left : w.right, at * tile, max_rows,
                                               max_cols, tile, step);
    const float x = (float)(c.item + c.step * heads_per_item * (b.hi - b.lo + 1));
    cost[keys ? t : n - 1 - t] = x;
    sum += x;
    most = std::max(most, (double)x);
  }
  if (n < n_tiles) {
    const double per_xcd = (nz * (double)num_heads + fa::kNumXcd - 1) / fa::kNumXcd, workers = std::max(1, num_cu / fa::kNumXcd);
    return std::max(sum / n * n_tiles * per_xcd / std::min(workers, n_tiles * per_xcd), most);
  }
  return fa::walk_time(fa::tile_work(nz * num_heads, zh_group, n_tiles), cost, n_tiles, num_cu);
}
bool wide_bwd_built(const fa_bwd_params* p, const Shape& s) {
  return !s.elementwise && is_16bit(p->Q.dtype) && s.d == 128 && !s.bias && !s.dropout && s.max_sq > 0 && s.max_sk > 0 && s.batch > 0;
}
BwdRoute bwd_route(const fa_bwd_params* p, const Shape& s, int num_cu) {
  BwdRoute r{false, false, false, 2, fa::q_head_group(s.hq, s.hk)};
  if (!wide_bwd_built(p, s)) return r;
  const int nz = s.num_seqlens != 0 ? std::abs(s.num_seqlens) : s.batch, group = s.hq / s.hk;
  constexpr int kLongest = 1 << 30;      // (the arithmetic on tiles goes a little past the end)
  const int max_sq = std::min(s.max_sq, kLongest), max_sk = std::min(s.max_sk, kLongest);
  int sq = max_sq, sk = max_sk;
  if (s.num_seqlens != 0) {
    const int share = s.num_seqlens > 0 ? nz : 1;
    sq = std::max(1, std::min(sq, (int)(p->Q.sizes[2] / share)));
    sk = std::max(1, std::min(sk, (int)(p->K.sizes[2] / share)));
  }
  struct Best { double t; int group; };
  auto walk = [&](bool keys, int tile, int step, WalkCost c) {
    const int heads = keys ? s.hk : s.hq, zg = keys ? 2 : fa::q_head_group(s.hq, s.hk), per_item = keys ? group : 1;
    const int rows = keys ? sk : sq, cols = keys ? sq : sk;
    Best b{tile_walk_time(p, s, keys, heads, zg, tile, step, per_item, c, num_cu, rows, cols, nz), zg};
    if (s.num_seqlens != 0) {
      const double longest = tile_walk_time(p, s, keys, 1, 1, tile, step, per_item, c, 1 << 20, keys ? max_sk : max_sq, keys ? max_sq : max_sk, 1);
      b.t = std::max(b.t, longest);
    } else if (tile == 256) {
      // all heads of an XCD side by side, the heavy tiles of all of them first: better balanced, more streams in flight
      const int all = (nz * heads + fa::kNumXcd - 1) / fa::kNumXcd;
      const double t = 1.04 * tile_walk_time(p, s, keys, heads, all, tile, step, per_item, c, num_cu, rows, cols, nz);
      if (t < b.t) b = Best{t, all};
    }
    return b;
  };
  const Best k_old = walk(true, 128, 64, {9, 1.95}), k_wide = walk(true, 256, 32, {7, 1.8});
  const Best q_old = walk(false, 128, 64, {5, 1.7}), q_wide = walk(false, 256, 32, {5, 1.42});
  // (with 128 rows half of every tile would be empty)
  r.wide_dkdv = sk > 128 && k_wide.t < k_old.t;
  r.wide_dq = sq > 128 && q_wide.t < q_old.t;
  r.group_dkdv = k_wide.group;
  r.group_dq = q_wide.group;
  // (keeping dS takes 0.9-1.1 of what the 128-row kernels take for recomputing)
  r.recompute = r.wide_dkdv && r.wide_dq && p->DB.ptr == nullptr && k_wide.t + q_wide.t < 0.97 * (k_old.t + q_old.t);
  return r;
}

// What of the stored dS (`need` bytes) and the parts fits `room` bytes of workspace, and the bytes it takes.  The
// parts give way first.
int64_t fit_workspace(int64_t room, int64_t* need, DkdvParts* parts) {
  if (*need > room) *need = 0;
  if (*need + parts->bytes > room) *parts = DkdvParts{1, 1, 0};
  return *need + parts->bytes;
}

}  // namespace

extern "C" {

const char* fa_get_name_suffix(void) { return "_amd_gfx950"; }
const char* fa_version(void) { return "0.1.0"; }

int fa_get_arch(void* hip_stream, char* buf, int32_t buflen) {
  const DeviceInfo* d = device_of_stream(static_cast<hipStream_t>(hip_stream));
  if (d == nullptr || buf == nullptr || buflen <= 0) return FA_ERROR_INVALID_VALUE;
  std::snprintf(buf, (size_t)buflen, "%s", d->arch);
  return FA_SUCCESS;
}

int fa_get_multiprocessor_count(void* hip_stream) {
  const DeviceInfo* d = device_of_stream(static_cast<hipStream_t>(hip_stream));
  return d ? d->num_cu : 40;   // v3src/util.cc:95-112 falls back to 40
}

int fa_get_clock_rate_khz(void* hip_stream) {
  const DeviceInfo* d = device_of_stream(static_cast<hipStream_t>(hip_stream));
  return d ? d->clock_khz : 0;
}

int fa_probe_mfma_rate(int32_t random_operands, int32_t num_workgroups, int32_t iters, float* out,
                       uint64_t* clocks, void* hip_stream) {
  if (out == nullptr || clocks == nullptr || num_workgroups <= 0 || iters <= 0) return FA_ERROR_INVALID_VALUE;
  hipStream_t stream = static_cast<hipStream_t>(hip_stream);
  const DeviceInfo* d = device_of_stream(stream);
  if (d == nullptr || !d->is_gfx950) return FA_ERROR_NO_BINARY_FOR_GPU;
  return (int)fa::run_mfma_rate(random_operands != 0, num_workgroups, iters, out,
                                reinterpret_cast<unsigned long long*>(clocks), stream);
}

int fa_write_words(void* dst, const uint32_t* words, int32_t count, void* hip_stream) {
  if (count < 0 || (count > 0 && (dst == nullptr || words == nullptr))) return FA_ERROR_INVALID_VALUE;
  return (int)fa::run_write_words(static_cast<uint32_t*>(dst), words, count, static_cast<hipStream_t>(hip_stream));
}

int fa_hip_get_last_error(void) { return (int)hipGetLastError(); }
int fa_hip_device_synchronize(void) { return (int)hipDeviceSynchronize(); }

int32_t fa_dropout_threshold(float dropout_p) { return fa::dropout_threshold(dropout_p); }

int fa_tile_intervals(int32_t causal_type, int32_t window_left, int32_t window_right, int32_t start_m,
                      int32_t seqlen_q, int32_t seqlen_k, int32_t block_m, int32_t block_n,
                      int32_t out[6]) {
  if (out == nullptr || block_m <= 0 || block_n <= 0) return FA_ERROR_INVALID_VALUE;
  const bool windowed = causal_type != 0;
  fa::Window w{0, 0};
  if (windowed) w = fa::parse_window(causal_type, window_left, window_right, seqlen_q, seqlen_k);
  const fa::BlockRanges r = fa::block_ranges(windowed, w.left, w.right, start_m, seqlen_q, seqlen_k,
                                             block_m, block_n);
  out[0] = r.lb_lo; out[1] = r.lb_hi; out[2] = r.fb_lo; out[3] = r.fb_hi; out[4] = r.rb_lo; out[5] = r.rb_hi;
  return FA_SUCCESS;
}

int fa_check_gpu(void* hip_stream) {
  const DeviceInfo* d = device_of_stream(static_cast<hipStream_t>(hip_stream));
  if (d == nullptr || !d->is_gfx950) return FA_ERROR_NO_BINARY_FOR_GPU;
  // the address of fa_attn_bwd_noalloc's array is looked up here as well: a first call of that
  // entry point under stream capture then finds it and makes no call that a capture forbids
  float* unused = nullptr;
  (void)scratch_of_device(device_index(d), &unused);
  return FA_SUCCESS;
}

int fa_validate_fwd(const fa_fwd_params* params, int32_t params_version, const fa_options* options) {
  return validate_fwd(params, params_version, options, nullptr);
}

int fa_validate_bwd(const fa_bwd_params* params, int32_t params_version, const fa_options* options) {
  return validate_bwd(params, params_version, options, nullptr, nullptr);
}

int fa_query_fwd_config(const fa_fwd_params* params, int32_t num_cu, fa_kernel_config* out) {
  if (out == nullptr) return FA_ERROR_INVALID_VALUE;
  Shape s{};
  int e = validate_fwd(params, FA_FWD_PARAMS_VERSION, nullptr, &s);
  if (e != FA_SUCCESS) return e;
  // the vector-ALU kernels (3-D grid), the fp32 kernels and the split-head-dim kernels (above 256)
  const bool valu = params->Q.dtype == FA_DTYPE_FLOAT32 || s.d > 256 || s.elementwise;
  const bool rows32 = !s.elementwise && params->Q.dtype == FA_DTYPE_FLOAT32 && f32_rows(s, false, params->causal_type, params->window_left, params->window_right, num_cu > 0 ? num_cu : 256);
  const int cus = num_cu > 0 ? num_cu : 256;
  const FwdPlan plan = fwd_plan(params->Q.dtype, s, params->causal_type, params->window_left, params->window_right, cus);
  const bool split = !plan.rows && plan.splits > 1;
  const bool may_wide = !plan.rows && fwd_wide(params, s, split ? plan.splits : 1, cus);
  const int half = split || plan.rows ? 0 : fwd_small_tiles(params, s, may_wide, cus);
  const bool wide = may_wide && !half;
  const fa::TileShape t = s.elementwise ? fa::TileShape{32, 1, 4, 0}
                          : rows32 ? fa::f32_rows_tile_shape(s.d)
                          : params->Q.dtype == FA_DTYPE_FLOAT32 ? fa::f32_tile_shape(s.d, -1)
                          : s.d > 256 ? fa::d512_tile_shape(-1)
                          : wide ? fa::fwd_wide_shape()
                                      : fa::fwd_tile_shape(params->Q.dtype, s.d, s.windowed, half);
  out->block_m = t.block_m; out->block_n = t.block_n; out->num_waves = t.num_waves;
  out->lds_bytes = t.lds_bytes;
  if (valu) {
    const int nz = s.num_seqlens != 0 ? std::abs(s.num_seqlens) : s.batch;
    const int mt = (s.max_sq + t.block_m - 1) / t.block_m;
    if (s.elementwise) {      // vector-ALU kernels: 3-D grid
      out->grid[0] = mt; out->grid[1] = s.hq; out->grid[2] = nz;
    } else if (rows32) {      // one workgroup per tile, the tiles of an XCD consecutive
      out->grid[0] = fa::kNumXcd * ((nz * s.hq * mt + fa::kNumXcd - 1) / fa::kNumXcd);
      out->grid[1] = 1; out->grid[2] = 1;
    } else {      // one workgroup per tile, the tiles of a kv-head's group back to back on one XCD
      out->grid[0] = fa::kNumXcd * ((nz * s.hk + fa::kNumXcd - 1) / fa::kNumXcd) * (s.hq / s.hk) * mt;
      out->grid[1] = 1; out->grid[2] = 1;
    }
  } else {
    const int nz = s.num_seqlens != 0 ? std::abs(s.num_seqlens) : s.batch;
    const fa::TileWork w = fa::tile_work(nz * s.hq, fa::q_head_group(s.hq, s.hk),
                                         (s.max_sq + t.block_m - 1) / t.block_m * (split ? plan.splits : 1));
    out->grid[0] = fa::kNumXcd * fa::tile_workers(w.items_per_xcd, cus, t.per_cu);
    out->grid[1] = 1;
    out->grid[2] = 1;
  }
  out->backend_index = 0;
  out->head_dim = s.d;
  out->flags = (s.windowed ? 1 : 0) | (s.bias ? 2 : 0) | (s.dropout ? 4 : 0) | (s.num_seqlens != 0 ? 8 : 0);
  // 64: the keys are split into parts, given scratch memory; 128: the packed-rows kernel takes the call (the tile and
  // grid above are those of the tile kernel)
  out->flags |= (plan.splits > 1 ? 64 : 0) | (plan.rows ? 128 : 0);
  // 32: fa_attn_fwd would run this call on packed copies in the workspace of the current device (the
  // tile and grid above are those of the element-wise kernels it runs on otherwise)
  int dev = 0;
  if (s.elementwise && hipGetDevice(&dev) == hipSuccess && dev >= 0 && dev < kMaxDevices &&
      (int64_t)fwd_copies_bytes(params) <= ws_limit_bytes(dev))
    out->flags |= 32;
  return FA_SUCCESS;
}

int fa_query_bwd_config(const fa_bwd_params* params, const fa_options* options, int32_t kernel_slot,
                        fa_kernel_config* out) {
  if (out == nullptr || kernel_slot < 0 || kernel_slot > 3) return FA_ERROR_INVALID_VALUE;
  Shape s{};
  int be = 0;
  int e = validate_bwd(params, FA_BWD_PARAMS_VERSION, options, &s, &be);
  if (e != FA_SUCCESS) return e;
  const bool valu = params->Q.dtype == FA_DTYPE_FLOAT32 || s.d > 256 || s.elementwise;   // vector-ALU kernels: 32 rows per workgroup
  if (valu && kernel_slot == 3) return FA_ERROR_PEER_ACCESS_UNSUPPORTED;
  const bool split_d = !s.elementwise && params->Q.dtype != FA_DTYPE_FLOAT32 && s.d > 256 && kernel_slot != 0;
  const bool f32_mfma = !s.elementwise && params->Q.dtype == FA_DTYPE_FLOAT32 && kernel_slot != 0;
  const bool rows32 = f32_mfma && f32_rows(s, true, params->causal_type, params->window_left, params->window_right, 256);
  constexpr int kCus = 256;      // assumed here
  const BwdRoute route = bwd_route(params, s, kCus);
  // what of the workspace's uses the call gets (a host without a device: no limit unless one was set)
  int ntq = 0, ntk = 0, dev = 0;
  int64_t ds_bytes = 0, stat_bytes = 0, need = 0;
  DkdvParts parts{1, 1, 0};
  const bool have_dev = hipGetDevice(&dev) == hipSuccess && dev >= 0 && dev < kMaxDevices;
  const int64_t set = g_ws_limit.load(std::memory_order_relaxed);
  if (be == 0) {
    need = ds_workspace_need(params, s, &ntq, &ntk, &ds_bytes, &stat_bytes);
    const int64_t room = have_dev ? ws_limit_bytes(dev) : set >= 0 ? set : INT64_MAX;
    parts = dkdv_parts(params, s, need > 0 && need <= room, kCus);
    if (route.recompute) {
      need = 0;
      parts = DkdvParts{1, 1, 0};
    }
    fit_workspace(room, &need, &parts);
  }
  const bool wide_dkdv = route.wide_dkdv && need == 0 && parts.bytes == 0;
  fa::BwdArgs a{};
  bias_args(*params, s, &a);
  a.seq = seq_args(s, params->cu_seqlens_q, params->cu_seqlens_k, params->seq_strides_q, params->seq_strides_k, params->varlen_type);
  const bool pair_dkdv = fa::bwd_dkdv_by_pairs(a, s.d, s.bias, need > 0);
  const fa::TileShape t = rows32 ? fa::f32_rows_tile_shape(s.d)
                          : f32_mfma ? fa::f32_tile_shape(s.d, kernel_slot)
                          : split_d ? fa::d512_tile_shape(kernel_slot)
                          : valu  ? (kernel_slot == 1 ? fa::TileShape{1, 32, 4, 0} : fa::TileShape{32, 1, 4, 0})
                          : kernel_slot == 1 && wide_dkdv ? fa::bwd_wide_shape(true)
                          : kernel_slot == 1 && pair_dkdv ? fa::bwd_pair_shape(s.bias)
                          : kernel_slot == 2 && route.wide_dq ? fa::bwd_wide_shape(false)
                                  : fa::bwd_tile_shape(params->Q.dtype, s.d, s.windowed, s.bias, s.dropout, kernel_slot, need > 0);
  const int nz = s.num_seqlens != 0 ? std::abs(s.num_seqlens) : s.batch;
  out->block_m = t.block_m; out->block_n = t.block_n; out->num_waves = t.num_waves;
  out->lds_bytes = t.lds_bytes;
  const int mt = (s.max_sq + t.block_m - 1) / t.block_m, nt = (s.max_sk + t.block_n - 1) / t.block_n;
  const int ratio = s.hq / s.hk;
  // 1-D work lists of the main kernels
  auto workers = [&](int heads, int zg, int items) {
    const fa::TileWork w = fa::tile_work(nz * heads, zg, items);
    return fa::kNumXcd * fa::bwd_workers(s.d, s.bias, w.items_per_xcd, kCus, t.per_cu);
  };
  out->grid[1] = 1;
  out->grid[2] = 1;
  if (rows32) {
    const int items = kernel_slot == 1 ? nz * s.hk * nt : nz * s.hq * mt;
    out->grid[0] = fa::kNumXcd * ((items + fa::kNumXcd - 1) / fa::kNumXcd);
  } else if (f32_mfma || split_d) {      // one workgroup per tile, the tiles of a kv-head back to back on one XCD
    out->grid[0] = fa::kNumXcd * ((nz * s.hk + fa::kNumXcd - 1) / fa::kNumXcd) * (kernel_slot == 1 ? nt : ratio * mt);
  } else if (valu) {
    out->grid[0] = kernel_slot == 1 ? nt : mt;
    out->grid[1] = kernel_slot == 1 ? s.hk : s.hq;
    out->grid[2] = nz;
  } else switch (kernel_slot) {
    case 0: out->grid[0] = mt; out->grid[1] = s.hq; out->grid[2] = nz; break;
    case 1: out->grid[0] = workers(s.hk, wide_dkdv ? route.group_dkdv : 2, nt * parts.heads * parts.tiles); break;
    case 2: out->grid[0] = workers(s.hq, route.wide_dq ? route.group_dq : fa::q_head_group(s.hq, s.hk), mt); break;
    default: out->grid[0] = workers(s.hk, 2, nt + mt * ratio); break;
  }
  out->backend_index = be;
  out->head_dim = s.d;
  out->flags = (s.windowed ? 1 : 0) | (s.bias ? 2 : 0) | (s.dropout ? 4 : 0) | (s.num_seqlens != 0 ? 8 : 0);
  // 16: fa_attn_bwd would keep dS in HBM for this call on the current device (workspace within the
  // limit; a call under stream capture recomputes all the same); 64: it would cut the dK/dV items into parts
  if (need > 0 && have_dev) out->flags |= 16;
  if (parts.bytes > 0) out->flags |= 64;
  // 32: fa_attn_bwd would run this call on packed copies in the workspace
  if (s.elementwise && have_dev && (int64_t)bwd_copies_bytes(params) <= ws_limit_bytes(dev)) out->flags |= 32;
  return FA_SUCCESS;
}

int fa_debug_simulate_encoded_softmax(const fa_tensor4* r, float dropout_p, const fa_tensor0* philox_seed,
                                      const fa_tensor0* philox_offset1, uint64_t philox_offset2,
                                      void* hip_stream) {
  if (r == nullptr || r->ptr == nullptr || philox_seed == nullptr || philox_offset1 == nullptr)
    return FA_ERROR_INVALID_VALUE;
  if (r->dtype != FA_DTYPE_FLOAT16 && r->dtype != FA_DTYPE_BFLOAT16 && r->dtype != FA_DTYPE_FLOAT32)
    return FA_ERROR_INVALID_VALUE;
  if (r->strides[3] != 1) return FA_ERROR_NOT_SUPPORTED;
  hipStream_t stream = static_cast<hipStream_t>(hip_stream);
  const DeviceInfo* d = device_of_stream(stream);
  if (d == nullptr || !d->is_gfx950) return FA_ERROR_NO_BINARY_FOR_GPU;
  fa::EncodedSoftmaxArgs a{};
  a.r = r->ptr;
  a.s_z = (int64_t)r->strides[0]; a.s_h = (int64_t)r->strides[1]; a.s_m = (int64_t)r->strides[2];
  a.batch = (int)r->sizes[0]; a.heads = (int)r->sizes[1];      // attn_debug.cc:40-42
  a.seqlen_q = (int)r->sizes[2]; a.seqlen_k = (int)r->sizes[3];
  a.dtype = r->dtype;
  a.drop = dropout_args(dropout_p, *philox_seed, *philox_offset1, philox_offset2);
  return (int)fa::run_encoded_softmax(a, stream);
}

static int attn_fwd_impl(const fa_fwd_params* p, int32_t params_version, void* hip_stream,
                         const fa_options* options, fa_allocator* alloc, bool key_mask = false) {
  Shape s{};
  int e = validate_fwd(p, params_version, options, &s);
  if (e != FA_SUCCESS) return e;
  if (key_mask && (s.elementwise || !is_16bit(p->Q.dtype) || s.d > 128 || s.dropout || s.num_seqlens != 0)) return FA_ERROR_NOT_SUPPORTED;
  hipStream_t stream = static_cast<hipStream_t>(hip_stream);
  const DeviceInfo* dev = device_of_stream(stream);
  if (dev == nullptr || !dev->is_gfx950) return FA_ERROR_NO_BINARY_FOR_GPU;

  if (s.elementwise && !t_ws_nested.active && !stream_is_capturing(stream)) {
    // packed copies of Q, K, V and Out in the workspace, the MFMA kernels on those, Out copied back
    const fa_tensor4* in[3] = {&p->Q, &p->K, &p->V};
    const size_t need = fwd_copies_bytes(p);
    void* base = nullptr;
    if ((int64_t)need <= ws_limit_bytes(device_index(dev)) && ws_acquire(device_index(dev), need, stream, &base) == hipSuccess) {
      fa_fwd_params p2 = *p;
      char* at = static_cast<char*>(base);
      fa_tensor4* to[3] = {&p2.Q, &p2.K, &p2.V};
      hipError_t err = hipSuccess;
      for (int i = 0; i < 3 && err == hipSuccess; ++i) {
        *to[i] = packed_view(*in[i], at);
        at += packed_bytes(*in[i]);
        err = repack(*in[i], *to[i], false, stream);
      }
      p2.Out = packed_view(p->Out, at);
      int rc = (int)err;
      if (err == hipSuccess) {
        t_ws_nested = NestedWorkspace{true, nullptr, 0};
        rc = attn_fwd_impl(&p2, params_version, hip_stream, options, alloc);
        t_ws_nested = NestedWorkspace{};
      }
      if (rc == FA_SUCCESS) rc = (int)repack(p->Out, p2.Out, true, stream);
      ws_release(device_index(dev), stream);
      return rc;
    }
  }

  fa::FwdArgs a{};
  a.q = p->Q.ptr; a.k = p->K.ptr; a.v = p->V.ptr; a.bias = p->B.ptr;
  a.out = p->Out.ptr;
  a.lse = static_cast<float*>(p->L.ptr);
  a.sq = strides3(p->Q); a.sk = strides3(p->K); a.sv = strides3(p->V); a.so = strides3(p->Out);
  if (s.bias) {
    a.sb_z = (int64_t)p->B.strides[0]; a.sb_h = (int64_t)p->B.strides[1];
    a.sb_m = (int64_t)p->B.strides[2]; a.sb_n = (int64_t)p->B.strides[3];
  }
  a.batch = s.batch; a.hq = s.hq; a.hk = s.hk; a.head_dim = s.d_qk; a.head_dim_v = s.d_v;
  a.elementwise = s.elementwise ? 1 : 0;
  a.sm_scale = p->Sm_scale;
  a.seq = seq_args(s, p->cu_seqlens_q, p->cu_seqlens_k, p->seq_strides_q, p->seq_strides_k, p->varlen_type);
  a.mask = fa::MaskArgs{p->causal_type, p->window_left, p->window_right};
  a.drop = dropout_args(p->dropout_p, p->philox_seed_ptr, p->philox_offset1, p->philox_offset2);
  a.seed_out = static_cast<uint64_t*>(p->philox_seed_output.ptr);
  a.offset_out = static_cast<uint64_t*>(p->philox_offset_output.ptr);
  a.atomic_counter = static_cast<int32_t*>(p->persistent_atomic_counter.ptr);
  a.num_cu = dev->num_cu;

  hipError_t err;
  const FwdPlan plan = fwd_plan(p->Q.dtype, s, p->causal_type, p->window_left, p->window_right, dev->num_cu);
  if (key_mask && !plan.rows && plan.splits > 1) return FA_ERROR_NOT_SUPPORTED;      // (split tiles take any bias as one of rows)
  a.key_mask = key_mask ? 1 : 0;
  void* scratch = nullptr;
  bool held = false;
  if (plan.splits > 1) {
    if (alloc != nullptr) {
      scratch = alloc->alloc(alloc, (uint64_t)plan.bytes);
    } else if (!t_ws_nested.active && !stream_is_capturing(stream) && plan.bytes <= ws_limit_bytes(device_index(dev))) {
      held = ws_acquire(device_index(dev), (size_t)plan.bytes, stream, &scratch) == hipSuccess;
      if (!held) scratch = nullptr;
    }
    if (scratch != nullptr) {
      a.part_o = static_cast<float*>(scratch);
      a.part_ml = reinterpret_cast<float*>(static_cast<char*>(scratch) + plan.o_bytes);
    }
  }
  a.splits = scratch != nullptr ? plan.splits : 1;
  const bool may_wide = !plan.rows && fwd_wide(p, s, a.splits, dev->num_cu);
  if (a.splits <= 1 && !plan.rows) a.half_tiles = fwd_small_tiles(p, s, may_wide, dev->num_cu);
  const bool wide = may_wide && !a.half_tiles;
  FA_LOG(4, "attn_fwd: D=%d windowed=%d bias=%d dropout=%d nseq=%d rows=%d splits=%d half_tiles=%d wide=%d", s.d, (int)s.windowed,
         (int)s.bias, (int)s.dropout, s.num_seqlens, (int)plan.rows, a.splits, a.half_tiles, (int)wide);
  if (plan.rows) {
    a.row_blocks = plan.row_blocks; a.part_rows = plan.part_rows;
    err = run_fwd_rows(p->Q.dtype, s.d, a, s, stream);
  } else if (wide) {
    err = fa::run_fwd_wide(p->Q.dtype, a, s.windowed, stream);
  } else {
    err = run_fwd(p->Q.dtype, s.d, a, s, stream);
  }
  if (held) ws_release(device_index(dev), stream);
  if (err != hipSuccess) return (int)err;
  if (p->encoded_softmax.ptr != nullptr) {
    // the forward metro chains the mask dump (modules/flash/aot/__init__.py:40-41)
    fa_tensor4 r = p->encoded_softmax;
    return fa_debug_simulate_encoded_softmax(&r, p->dropout_p, &p->philox_seed_ptr, &p->philox_offset1,
                                             p->philox_offset2, hip_stream);
  }
  return FA_SUCCESS;
}

int fa_attn_fwd(const fa_fwd_params* p, int32_t params_version, void* hip_stream, const fa_options* options) {
  return attn_fwd_impl(p, params_version, hip_stream, options, nullptr);
}

int fa_attn_fwd_alloc(const fa_fwd_params* p, int32_t params_version, void* hip_stream, const fa_options* options,
                      fa_allocator* alloc) {
  return attn_fwd_impl(p, params_version, hip_stream, options, alloc);
}

int fa_attn_fwd_key_mask(const fa_fwd_params* p, int32_t params_version, void* hip_stream, const fa_options* options,
                         fa_allocator* alloc) {
  if (p == nullptr || p->B.ptr == nullptr || p->B.dtype != FA_DTYPE_UINT8) return FA_ERROR_INVALID_VALUE;
  if (p->B.sizes[2] > 1 && p->B.strides[2] != 0) return FA_ERROR_NOT_SUPPORTED;
  fa_fwd_params q = *p;
  q.B.dtype = p->Q.dtype;
  q.B.strides[2] = 0;
  return attn_fwd_impl(&q, params_version, hip_stream, options, alloc, true);
}

// kernel_slot < 0: the whole backward of the chosen backend; otherwise only that
// kernel (0 delta, 1 dK/dV, 2 dQ, 3 fused; 4-6 the three kernels of the backward that keeps dS).
// own_delta: the split backend with delta in the library's own per-device array (params->D is
// not looked at).
static int attn_bwd_impl(const fa_bwd_params* p_in, int32_t params_version, void* hip_stream,
                         const fa_options* options, int kernel_slot, bool own_delta = false) {
  Shape s{};
  int backend = 0;
  fa_options forced{};
  const fa_bwd_params* p = p_in;
  fa_bwd_params with_delta;
  if (own_delta) {
    if (p_in == nullptr) return FA_ERROR_INVALID_VALUE;
    if (params_version != FA_BWD_PARAMS_VERSION) return FA_ERROR_INVALID_SYMBOL;
    hipStream_t st = static_cast<hipStream_t>(hip_stream);
    const DeviceInfo* dv = device_of_stream(st);
    if (dv == nullptr || !dv->is_gfx950) return FA_ERROR_NO_BINARY_FOR_GPU;
    float* ptr = nullptr;
    hipError_t se = scratch_of_device(device_index(dv), &ptr);
    if (se != hipSuccess) return (int)se;
    with_delta = *p_in;
    with_delta.D = fa_lazy_tensor2{};
    with_delta.D.eager.ptr = ptr;
    // sized for the check of the tensors below; the limit of the array is tested right after
    with_delta.D.eager.sizes[0] = 1; with_delta.D.eager.sizes[1] = (uint64_t)1 << 60;
    with_delta.D.eager.strides[0] = (uint64_t)1 << 60; with_delta.D.eager.strides[1] = 1;
    with_delta.D.eager.dtype = FA_DTYPE_FLOAT32;
    p = &with_delta;
    forced.force_backend_index = 0;
    forced.deterministic = 0;
    options = &forced;
    Shape probe{};
    const int pe = validate_bwd(p, params_version, options, &probe, nullptr);
    if (pe != FA_SUCCESS) return pe;
    // one delta value per (batch element or token, query head, query row)
    if (probe.row_stats > kScratchFloats) {
      FA_LOG(1, "attn_bwd_noalloc: %lld delta values needed, the library's array holds %lld",
             (long long)probe.row_stats, (long long)kScratchFloats);
      return FA_ERROR_OUT_OF_MEMORY;
    }
  }
  if (kernel_slot >= 0) {
    forced.force_backend_index = kernel_slot == 3 ? 1 : 0;   // (slots 4-6 belong to the split backend too)
    forced.deterministic = 0;
    options = &forced;
  }
  int e = validate_bwd(p, params_version, options, &s, &backend);
  if (e != FA_SUCCESS) return e;
  hipStream_t stream = static_cast<hipStream_t>(hip_stream);
  const DeviceInfo* dev = device_of_stream(stream);
  if (dev == nullptr || !dev->is_gfx950) return FA_ERROR_NO_BINARY_FOR_GPU;

  if (s.elementwise && kernel_slot < 0 && !own_delta && !t_ws_nested.active && !stream_is_capturing(stream)) {
    // packed copies of the eight activation tensors, the MFMA kernels on those, dQ, dK, dV copied back;
    // the packed call gets the rest of the buffer for its own use (dS)
    const fa_tensor4* all[8] = {&p->Q, &p->K, &p->V, &p->Out, &p->DO, &p->DQ, &p->DK, &p->DV};
    // (a call for backend 1 that will run the split kernels and brings no delta buffer gets one here)
    const bool lib_delta = backend == 1 && s.fused_as_split && p->D.eager.ptr == nullptr && p->D.acquire == nullptr;
    const size_t delta_bytes = lib_delta ? (((size_t)s.row_stats * 4 + 255) & ~(size_t)255) : 0;
    const size_t copies = bwd_copies_bytes(p) + delta_bytes;
    fa_bwd_params p2 = *p;
    fa_tensor4* to[8] = {&p2.Q, &p2.K, &p2.V, &p2.Out, &p2.DO, &p2.DQ, &p2.DK, &p2.DV};
    for (int i = 0; i < 8; ++i) *to[i] = packed_view(*all[i], reinterpret_cast<void*>(uintptr_t(256)));   // shapes first
    Shape s2{};
    int be2 = 0;
    int64_t inner = 0;
    if (validate_bwd(&p2, params_version, options, &s2, &be2) == FA_SUCCESS && be2 == 0) {
      int ntq = 0, ntk = 0;
      int64_t ds_bytes = 0, stat_bytes = 0;
      int64_t ds_need = ds_workspace_need(&p2, s2, &ntq, &ntk, &ds_bytes, &stat_bytes);
      const int64_t room = ws_limit_bytes(device_index(dev)) - (int64_t)copies;
      DkdvParts parts = dkdv_parts(&p2, s2, ds_need > 0 && ds_need <= room, dev->num_cu);
      inner = fit_workspace(room, &ds_need, &parts);
    }
    const size_t need = copies + (size_t)inner;
    void* base = nullptr;
    if ((int64_t)need <= ws_limit_bytes(device_index(dev)) && ws_acquire(device_index(dev), need, stream, &base) == hipSuccess) {
      char* at = static_cast<char*>(base);
      hipError_t err = hipSuccess;
      for (int i = 0; i < 8; ++i) {
        *to[i] = packed_view(*all[i], at);
        at += packed_bytes(*all[i]);
        if (i < 5 && err == hipSuccess) err = repack(*all[i], *to[i], false, stream);
      }
      if (lib_delta) {
        p2.D = fa_lazy_tensor2{};
        p2.D.eager = row_stats_view(at, s.row_stats);
        at += delta_bytes;
      }
      int rc = (int)err;
      if (err == hipSuccess) {
        t_ws_nested = NestedWorkspace{true, inner > 0 ? at : nullptr, (size_t)inner};
        rc = attn_bwd_impl(&p2, params_version, hip_stream, options, kernel_slot, false);
        t_ws_nested = NestedWorkspace{};
      }
      for (int i = 5; i < 8 && rc == FA_SUCCESS; ++i) rc = (int)repack(*all[i], *to[i], true, stream);
      ws_release(device_index(dev), stream);
      return rc;
    }
  }
  if (backend == 1 && s.fused_as_split) {
    // the split kernels: with the caller's delta buffer, or with one in the workspace
    if (kernel_slot == 3) return FA_ERROR_PEER_ACCESS_UNSUPPORTED;      // there is no such kernel to run alone
    if (p->D.eager.ptr != nullptr || p->D.acquire != nullptr) {
      backend = 0;
    } else {
      const size_t bytes = ((size_t)s.row_stats * 4 + 255) & ~(size_t)255;
      void* base = nullptr;
      if (kernel_slot >= 0 || t_ws_nested.active || stream_is_capturing(stream) ||
          (int64_t)bytes > ws_limit_bytes(device_index(dev)) ||
          ws_acquire(device_index(dev), bytes, stream, &base) != hipSuccess)
        return FA_ERROR_PEER_ACCESS_UNSUPPORTED;
      fa_bwd_params p2 = *p;
      p2.D = fa_lazy_tensor2{};
      p2.D.eager = row_stats_view(base, s.row_stats);
      fa_options split = options != nullptr ? *options : fa_options{};
      split.force_backend_index = 0;
      t_ws_nested = NestedWorkspace{true, nullptr, 0};
      const int rc = attn_bwd_impl(&p2, params_version, hip_stream, &split, -1, false);
      t_ws_nested = NestedWorkspace{};
      ws_release(device_index(dev), stream);
      return rc;
    }
  }
  if (s.elementwise && backend == 1) {
    // fused_without_copies: the element-wise kernels have the split backend only
    const bool forced = options != nullptr && options->force_backend_index >= 0;
    if (forced || (p->D.eager.ptr == nullptr && p->D.acquire == nullptr)) return FA_ERROR_PEER_ACCESS_UNSUPPORTED;
    if (p->D.eager.ptr != nullptr && (e = check_row_stats(p->D.eager, s.row_stats)) != FA_SUCCESS) return e;
    backend = 0;
  }

  fa::BwdArgs a{};
  a.q = p->Q.ptr; a.k = p->K.ptr; a.v = p->V.ptr;
  bias_args(*p, s, &a);
  a.out = p->Out.ptr; a.dout = p->DO.ptr;
  a.dq = p->DQ.ptr; a.dk = p->DK.ptr; a.dv = p->DV.ptr; a.db = p->DB.ptr;
  a.lse = static_cast<const float*>(p->L.ptr);
  a.sq = strides3(p->Q); a.sk = strides3(p->K); a.sv = strides3(p->V); a.so = strides3(p->Out);
  a.sdo = strides3(p->DO); a.sdq = strides3(p->DQ); a.sdk = strides3(p->DK); a.sdv = strides3(p->DV);
  if (p->DB.ptr != nullptr) {
    a.sdb_z = (int64_t)p->DB.strides[0]; a.sdb_h = (int64_t)p->DB.strides[1];
    a.sdb_m = (int64_t)p->DB.strides[2]; a.sdb_n = (int64_t)p->DB.strides[3];
  }
  a.batch = s.batch; a.hq = s.hq; a.hk = s.hk; a.head_dim = s.d_qk; a.head_dim_v = s.d_v;
  a.elementwise = s.elementwise ? 1 : 0;
  a.sm_scale = p->Sm_scale;
  a.seq = seq_args(s, p->cu_seqlens_q, p->cu_seqlens_k, p->seq_strides_q, p->seq_strides_k, p->varlen_type);
  a.mask = fa::MaskArgs{p->causal_type, p->window_left, p->window_right};
  a.drop = dropout_args(p->dropout_p, p->philox_seed_ptr, p->philox_offset1, p->philox_offset2);
  a.num_cu = dev->num_cu;

  const int dt = p->Q.dtype;
  FA_LOG(4, "attn_bwd: backend=%d slot=%d D=%d windowed=%d bias=%d dropout=%d nseq=%d", backend,
         kernel_slot, s.d, (int)s.windowed, (int)s.bias, (int)s.dropout, s.num_seqlens);
  hipError_t err = hipSuccess;
  if (backend == 0) {
    // split: delta, then dK/dV, then dQ (modules/flash/aot/__init__.py:52-59)
    fa_lazy_tensor2* lazy = const_cast<fa_lazy_tensor2*>(&p->D);
    fa_tensor2 delta = p->D.eager;
    bool acquired = false;
    if (delta.ptr == nullptr) {
      const bool no_query = p->Q.sizes[0] == 0 || p->Q.sizes[2] == 0;
      if (lazy->acquire(lazy, &delta) != 0 || (delta.ptr == nullptr && !no_query)) return FA_ERROR_INVALID_VALUE;
      acquired = true;
      if (delta.ptr != nullptr && check_row_stats(delta, s.row_stats) != FA_SUCCESS) {
        if (lazy->dispose != nullptr) lazy->dispose(lazy);
        return FA_ERROR_INVALID_VALUE;
      }
    }
    a.delta = static_cast<float*>(delta.ptr);
    const bool slow = s.elementwise;              // rows moved element by element: vector-ALU kernels
    const bool f32 = !slow && dt == FA_DTYPE_FLOAT32;      // fp32 MFMA kernels
    const bool big = !slow && !f32 && s.d > 256;  // head dim split over the waves
    // fp32 and the head dims above 256 take delta from the vector-ALU kernel.  The dQ kernel of the
    // 16-bit types up to head dim 256 computes delta from the O and dO rows it holds and writes it
    // out; the dK/dV kernel runs after it and reads it, so the whole backward is two launches
    // (kernel_slot 0 still launches the preprocess kernel on its own).
    // (fa_f32_rows.hip does the same)
    const bool rows32 = f32 && f32_rows(s, true, p->causal_type, p->window_left, p->window_right, dev->num_cu);
    const bool delta_launch = (f32 && !rows32) || big || slow;
    // The 16-bit kernels up to head dim 256 can keep dS in HBM instead of recomputing S and dP in
    // the dQ kernel (5 GEMMs instead of 7): delta first, then dK/dV writing dS, then dQ = dS K.  It
    // takes 2 bytes per (query, key) pair of workspace; when that is above the limit, under stream
    // capture, for packed sequences and where ds_workspace_need says so the kernels recompute.  (Measured at S4096, 16384 tokens:
    // head dim 128 gains 5 %, 256 gains 16 %; head dim 64, where a pair costs half the arithmetic and
    // the same bytes, loses 12 % unless the dQ kernel is spared dropout or a bias: then it gains 20-30 %.)
    void* ds_ws = nullptr;
    int ntq = 0, ntk = 0;
    int64_t ds_bytes = 0, stat_bytes = 0;
    // (kernel_slot 4, 5, 6: one kernel of this backward only; the buffer keeps its content between calls)
    const int ds_slot = kernel_slot >= 4 ? kernel_slot - 4 : -1;
    int64_t need = (kernel_slot < 0 || ds_slot >= 0) && !own_delta
                       ? ds_workspace_need(p, s, &ntq, &ntk, &ds_bytes, &stat_bytes) : 0;
    const int64_t limit = ws_limit_bytes(device_index(dev));
    if (ds_slot >= 0 && (need == 0 || need > limit)) {
      if (acquired && lazy->dispose != nullptr) lazy->dispose(lazy);
      return FA_ERROR_NOT_SUPPORTED;
    }
    // a nested call: the caller holds the buffer and has set a part of it aside
    const bool nested = t_ws_nested.active;
    const int64_t room = nested ? (int64_t)t_ws_nested.bytes : limit;
    // (single kernels, for timing, run uncut)
    DkdvParts parts{1, 1, 0};
    if (kernel_slot < 0 && !own_delta) parts = dkdv_parts(p, s, need > 0 && need <= room, dev->num_cu);
    const BwdRoute route = bwd_route(p, s, dev->num_cu);
    if (route.recompute && kernel_slot < 0) {
      need = 0;
      parts = DkdvParts{1, 1, 0};
    }
    int64_t bytes = fit_workspace(room, &need, &parts);
    void* ws = nested ? t_ws_nested.ptr : nullptr;
    bool held = false;
    if (!nested && bytes > 0 && !stream_is_capturing(stream)) {
      held = ws_acquire(device_index(dev), (size_t)bytes, stream, &ws) == hipSuccess;
      if (!held && need > 0 && need < bytes) {      // no memory for both
        bytes = fit_workspace(need, &need, &parts);
        held = ws_acquire(device_index(dev), (size_t)bytes, stream, &ws) == hipSuccess;
      }
      if (!held) {
        ws = nullptr;
        FA_LOG(2, "attn_bwd: no workspace of %lld bytes, recomputing instead", (long long)bytes);
      }
    }
    if (ws != nullptr && need > 0) {
      ds_ws = ws;
      a.ds_ntq = ntq;
      a.ds_ntk = ntk;
      a.lse_scaled = reinterpret_cast<const float*>(static_cast<char*>(ds_ws) + ds_bytes);
      a.delta_prep = reinterpret_cast<const float*>(static_cast<char*>(ds_ws) + ds_bytes + stat_bytes);
    }
    const bool cut = ws != nullptr && parts.bytes > 0;
    if (cut) {
      a.part_heads = parts.heads; a.part_tiles = parts.tiles;
      a.part_ws = reinterpret_cast<float*>(static_cast<char*>(ws) + need);
    }
    auto run_dkdv = [&]() {
      if (route.wide_dkdv && !cut && a.ds_ws == nullptr) {
        a.walk_group = route.group_dkdv;
        return fa::run_bwd_dkdv_wide(dt, a, s.windowed, stream);
      }
      if (fa::bwd_dkdv_by_pairs(a, s.d, s.bias, a.ds_ws != nullptr))
        return fa::run_bwd_dkdv_pair(dt, a, s.windowed, s.bias, s.dropout, stream);
      return (cut ? fa::run_bwd_dkdv_parts : fa::run_bwd_dkdv)(dt, s.d, a, s.windowed, s.bias, s.dropout, stream);
    };
    if (ds_slot >= 0 && ds_ws == nullptr) {
      if (acquired && lazy->dispose != nullptr) lazy->dispose(lazy);
      return FA_ERROR_NOT_SUPPORTED;          // under stream capture, or no memory
    }
    if (ds_ws != nullptr) {
      if (ds_slot < 0 || ds_slot == 0) err = fa::run_bwd_preprocess(dt, s.d, a, stream);
      a.ds_ws = ds_ws;
      if (err == hipSuccess && (ds_slot < 0 || ds_slot == 1))
        err = run_dkdv();
      if (err == hipSuccess && (ds_slot < 0 || ds_slot == 2)) err = fa::run_bwd_dqs(dt, s.d, a, stream);
      if (held) ws_release(device_index(dev), stream);
      if (acquired && lazy->dispose != nullptr) lazy->dispose(lazy);
      return (int)err;
    }
    if (kernel_slot == 0 || (kernel_slot < 0 && delta_launch))
      err = delta_launch || f32 ? fa::run_bwd_valu(dt, s.d, 0, a, stream) : fa::run_bwd_preprocess(dt, s.d, a, stream);
    const int order[2] = {delta_launch ? 1 : 2, delta_launch ? 2 : 1};
    for (int i = 0; i < 2 && err == hipSuccess; ++i) {
      const int slot = order[i];
      if (kernel_slot >= 0 && kernel_slot != slot) continue;
      if (slow)
        err = fa::run_bwd_valu(dt, s.d, slot, a, stream);
      else if (f32)
        err = (rows32 ? fa::run_bwd_f32_rows : fa::run_bwd_f32)(s.d, slot, a, s.windowed, s.bias, s.dropout, stream);
      else if (big)
        err = fa::run_bwd_d512(dt, slot, a, s.windowed, s.bias, s.dropout, stream);
      else if (slot == 1)
        err = run_dkdv();
      else if (route.wide_dq) {
        a.walk_group = route.group_dq;
        err = fa::run_bwd_dq_wide(dt, a, s.windowed, stream);
      } else
        err = fa::run_bwd_dq(dt, s.d, a, s.windowed, s.bias, s.dropout, stream);
    }
    if (held) ws_release(device_index(dev), stream);
    if (acquired && lazy->dispose != nullptr) lazy->dispose(lazy);   // attn_bwd.cc:157
  } else {
    a.delta = nullptr;
    err = fa::run_bwd_fused(dt, s.d, a, s.windowed, s.bias, s.dropout, stream);
  }
  return (int)err;
}

int fa_attn_bwd(const fa_bwd_params* p, int32_t params_version, void* hip_stream,
                const fa_options* options) {
  return attn_bwd_impl(p, params_version, hip_stream, options, -1);
}

// ---- v2 positional entry points ------------------------------------------------------------
// Thin fills of the v3 params: is_causal -> windowed with the top-left sentinels, compact
// packed sequences -> varlen_type 1 (the reference's Python layer does the same,
// modules/flash/tests/aotriton_flash.py:141-196,277-335).

extern "C++" {
namespace {
template <typename V> V view_or_null(const V* t) { return t ? *t : V{}; }

void set_causal(bool is_causal, int8_t* type, int32_t* left, int32_t* right) {
  *type = is_causal ? FA_CAUSAL_WINDOWED : FA_CAUSAL_NONE;
  *left = *right = is_causal ? FA_WINDOW_TOP_LEFT : 0;
}

int v2_fwd(const fa_tensor4* q, const fa_tensor4* k, const fa_tensor4* v, const fa_tensor4* b,
           const fa_tensor1* cu_q, const fa_tensor1* cu_k, int32_t max_sq, int32_t max_sk, float sm_scale,
           const fa_tensor2* lse, const fa_tensor4* out, float dropout_p, const fa_tensor0* seed,
           const fa_tensor0* off1, int64_t off2, const fa_tensor0* seed_out, const fa_tensor0* off_out,
           const fa_tensor4* encoded_softmax, int32_t is_causal, const fa_tensor0* atomic, void* stream) {
  if (q == nullptr || k == nullptr || v == nullptr || out == nullptr) return FA_ERROR_INVALID_VALUE;
  fa_fwd_params p{};
  p.Q = *q; p.K = *k; p.V = *v; p.B = view_or_null(b);
  p.Sm_scale = sm_scale;
  p.L = view_or_null(lse);
  p.Out = *out;
  p.cu_seqlens_q = view_or_null(cu_q); p.cu_seqlens_k = view_or_null(cu_k);
  p.Max_seqlen_q = max_sq; p.Max_seqlen_k = max_sk;
  p.varlen_type = cu_q != nullptr ? FA_VARLEN_COMPACT : FA_VARLEN_NONE;
  p.dropout_p = dropout_p;
  p.philox_seed_ptr = view_or_null(seed); p.philox_offset1 = view_or_null(off1);
  p.philox_offset2 = (uint64_t)off2;
  p.philox_seed_output = view_or_null(seed_out); p.philox_offset_output = view_or_null(off_out);
  p.encoded_softmax = view_or_null(encoded_softmax);
  p.persistent_atomic_counter = view_or_null(atomic);
  set_causal(is_causal != 0, &p.causal_type, &p.window_left, &p.window_right);
  return fa_attn_fwd(&p, FA_FWD_PARAMS_VERSION, stream, nullptr);
}

int v2_bwd(const fa_tensor4* q, const fa_tensor4* k, const fa_tensor4* v, const fa_tensor4* b,
           const fa_tensor1* cu_q, const fa_tensor1* cu_k, int32_t max_sq, int32_t max_sk, float sm_scale,
           const fa_tensor4* out, const fa_tensor4* dout, const fa_tensor4* dq, const fa_tensor4* dk,
           const fa_tensor4* dv, const fa_tensor4* db, const fa_tensor2* lse, const fa_tensor2* delta,
           float dropout_p, const fa_tensor0* seed, const fa_tensor0* off1, int64_t off2, int32_t is_causal,
           int backend, void* stream) {
  if (q == nullptr || k == nullptr || v == nullptr || out == nullptr || dout == nullptr || dq == nullptr ||
      dk == nullptr || dv == nullptr || lse == nullptr)
    return FA_ERROR_INVALID_VALUE;
  fa_bwd_params p{};
  p.Q = *q; p.K = *k; p.V = *v; p.B = view_or_null(b);
  p.Sm_scale = sm_scale;
  p.Out = *out; p.DO = *dout; p.DQ = *dq; p.DK = *dk; p.DV = *dv; p.DB = view_or_null(db);
  p.L = *lse;
  p.D.eager = view_or_null(delta);
  p.cu_seqlens_q = view_or_null(cu_q); p.cu_seqlens_k = view_or_null(cu_k);
  p.Max_seqlen_q = max_sq; p.Max_seqlen_k = max_sk;
  p.varlen_type = cu_q != nullptr ? FA_VARLEN_COMPACT : FA_VARLEN_NONE;
  p.dropout_p = dropout_p;
  p.philox_seed_ptr = view_or_null(seed); p.philox_offset1 = view_or_null(off1);
  p.philox_offset2 = (uint64_t)off2;
  set_causal(is_causal != 0, &p.causal_type, &p.window_left, &p.window_right);
  fa_options opt{backend, 0};
  return fa_attn_bwd(&p, FA_BWD_PARAMS_VERSION, stream, &opt);
}
}  // namespace
}  // extern "C++"

int fa_v2_attn_fwd(const fa_tensor4* q, const fa_tensor4* k, const fa_tensor4* v, const fa_tensor4* b,
                   float sm_scale, const fa_tensor2* softmax_lse, const fa_tensor4* out, float dropout_p,
                   const fa_tensor0* philox_seed, const fa_tensor0* philox_offset1, int64_t philox_offset2,
                   const fa_tensor0* philox_seed_output, const fa_tensor0* philox_offset_output,
                   const fa_tensor4* encoded_softmax, int32_t is_causal, const fa_tensor0* atomic_for_causal,
                   void* hip_stream) {
  return v2_fwd(q, k, v, b, nullptr, nullptr, 0, 0, sm_scale, softmax_lse, out, dropout_p, philox_seed,
                philox_offset1, philox_offset2, philox_seed_output, philox_offset_output, encoded_softmax,
                is_causal, atomic_for_causal, hip_stream);
}

int fa_v2_attn_fwd_compact_varlen(const fa_tensor4* q, const fa_tensor4* k, const fa_tensor4* v,
                                  const fa_tensor4* b, const fa_tensor1* cu_seqlens_q,
                                  const fa_tensor1* cu_seqlens_k, int32_t max_seqlen_q, int32_t max_seqlen_k,
                                  float sm_scale, const fa_tensor2* softmax_lse, const fa_tensor4* out,
                                  float dropout_p, const fa_tensor0* philox_seed,
                                  const fa_tensor0* philox_offset1, int64_t philox_offset2,
                                  const fa_tensor0* philox_seed_output, const fa_tensor0* philox_offset_output,
                                  const fa_tensor4* encoded_softmax, int32_t is_causal,
                                  const fa_tensor0* atomic_for_causal, void* hip_stream) {
  if (cu_seqlens_q == nullptr || cu_seqlens_k == nullptr) return FA_ERROR_INVALID_VALUE;
  return v2_fwd(q, k, v, b, cu_seqlens_q, cu_seqlens_k, max_seqlen_q, max_seqlen_k, sm_scale, softmax_lse, out,
                dropout_p, philox_seed, philox_offset1, philox_offset2, philox_seed_output, philox_offset_output,
                encoded_softmax, is_causal, atomic_for_causal, hip_stream);
}

int fa_v2_attn_bwd(const fa_tensor4* q, const fa_tensor4* k, const fa_tensor4* v, const fa_tensor4* b,
                   float sm_scale, const fa_tensor4* out, const fa_tensor4* dout, const fa_tensor4* dq,
                   const fa_tensor4* dk, const fa_tensor4* dv, const fa_tensor4* db,
                   const fa_tensor2* softmax_lse, const fa_tensor2* delta, float dropout_p,
                   const fa_tensor0* philox_seed, const fa_tensor0* philox_offset1, int64_t philox_offset2,
                   int32_t is_causal, void* hip_stream) {
  if (delta == nullptr) return FA_ERROR_INVALID_VALUE;
  return v2_bwd(q, k, v, b, nullptr, nullptr, 0, 0, sm_scale, out, dout, dq, dk, dv, db, softmax_lse, delta,
                dropout_p, philox_seed, philox_offset1, philox_offset2, is_causal, 0, hip_stream);
}

int fa_v2_attn_bwd_fused(const fa_tensor4* q, const fa_tensor4* k, const fa_tensor4* v, const fa_tensor4* b,
                         float sm_scale, const fa_tensor4* out, const fa_tensor4* dout, const fa_tensor4* dq,
                         const fa_tensor4* dk, const fa_tensor4* dv, const fa_tensor4* db,
                         const fa_tensor2* softmax_lse, float dropout_p, const fa_tensor0* philox_seed,
                         const fa_tensor0* philox_offset1, int64_t philox_offset2, int32_t is_causal,
                         void* hip_stream) {
  return v2_bwd(q, k, v, b, nullptr, nullptr, 0, 0, sm_scale, out, dout, dq, dk, dv, db, softmax_lse, nullptr,
                dropout_p, philox_seed, philox_offset1, philox_offset2, is_causal, 1, hip_stream);
}

int fa_v2_attn_bwd_compact_varlen(const fa_tensor4* q, const fa_tensor4* k, const fa_tensor4* v,
                                  const fa_tensor1* cu_seqlens_q, const fa_tensor1* cu_seqlens_k,
                                  int32_t max_seqlen_q, int32_t max_seqlen_k, const fa_tensor4* b, float sm_scale,
                                  const fa_tensor4* out, const fa_tensor4* dout, const fa_tensor4* dq,
                                  const fa_tensor4* dk, const fa_tensor4* dv, const fa_tensor4* db,
                                  const fa_tensor2* softmax_lse, const fa_tensor2* delta, float dropout_p,
                                  const fa_tensor0* philox_seed, const fa_tensor0* philox_offset1,
                                  int64_t philox_offset2, int32_t is_causal, void* hip_stream) {
  if (cu_seqlens_q == nullptr || cu_seqlens_k == nullptr || delta == nullptr) return FA_ERROR_INVALID_VALUE;
  return v2_bwd(q, k, v, b, cu_seqlens_q, cu_seqlens_k, max_seqlen_q, max_seqlen_k, sm_scale, out, dout, dq, dk,
                dv, db, softmax_lse, delta, dropout_p, philox_seed, philox_offset1, philox_offset2, is_causal, 0,
                hip_stream);
}

void fa_set_bwd_workspace_limit(int64_t bytes) { g_ws_limit.store(bytes, std::memory_order_relaxed); }

int fa_trim_workspace(void) {
  hipError_t err = hipSuccess;
  for (int d = 0; d < kMaxDevices; ++d) {
    std::lock_guard<std::mutex> lock(g_ws[d].mutex);
    if (g_ws[d].ptr != nullptr) {
      const hipError_t e = hipFree(g_ws[d].ptr);      // waits for the device first
      g_ws[d].ptr = nullptr; g_ws[d].bytes = 0; g_ws[d].used = g_ws[d].on_null = false;
      if (err == hipSuccess) err = e;
    }
  }
  return (int)err;
}

int fa_attn_bwd_noalloc(const fa_bwd_params* p, int32_t params_version, void* hip_stream) {
  return attn_bwd_impl(p, params_version, hip_stream, nullptr, -1, true);
}

int fa_attn_bwd_kernel(const fa_bwd_params* p, int32_t params_version, void* hip_stream,
                       int32_t kernel_slot) {
  if (kernel_slot < 0 || kernel_slot > 6) return FA_ERROR_INVALID_VALUE;
  return attn_bwd_impl(p, params_version, hip_stream, nullptr, kernel_slot);
}

}  // extern "C"
