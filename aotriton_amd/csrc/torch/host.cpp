// Native host path between PyTorch and the C ABI: what the Python layer does per call (tensor ->
// view marshalling, output allocation, Philox state, autograd bookkeeping), in one C++ call each.
//
// Small calls are bound by this path, not by the GPU: a forward on tensors of a few hundred KB takes
// 5-20 us on the device, where the ctypes layer needed 36 us for a forward, 53-64 us for a backward
// and the torch.library Python ops several times that (forward + backward of B8 H16 S512 D64 bf16
// through the SDPA entry point: 438 us per pass for 75 us of kernels).
//
// Three groups of functions:
//   attn_fwd, attn_bwd          the operator wrappers of aotriton_amd.flash (hipError_t as an int)
//   attention, attention_varlen the autograd Functions of aotriton_amd.autograd
//   sdpa_ops, sdpa_function     F.scaled_dot_product_attention-shaped, on the custom ops / on `attention`
// and the registration of the custom ops torch.ops.aotriton_amd.* (fake implementations are in
// torch_ops.py).
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/core/dispatch/Dispatcher.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/forward_grad.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/pybind.h>
#include <torch/library.h>

#include <cmath>
#include <limits>
#include <optional>
#include <string>
#include <tuple>
#include <vector>

#include "aotriton_amd/flash.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// ---- views ------------------------------------------------------------------------------------

int dtype_code(at::ScalarType t) {
  switch (t) {
    case at::kFloat: return FA_DTYPE_FLOAT32;
    case at::kHalf: return FA_DTYPE_FLOAT16;
    case at::kBFloat16: return FA_DTYPE_BFLOAT16;
    case at::kChar: return FA_DTYPE_INT8;
    case at::kShort: return FA_DTYPE_INT16;
    case at::kInt: return FA_DTYPE_INT32;
    case at::kLong: return FA_DTYPE_INT64;
    case at::kByte: return FA_DTYPE_UINT8;
    case at::kUInt16: return FA_DTYPE_UINT16;
    case at::kUInt32: return FA_DTYPE_UINT32;
    case at::kUInt64: return FA_DTYPE_UINT64;
    default: return FA_DTYPE_UNKNOWN;
  }
}

// View of a tensor of rank N (fa_tensor4, fa_tensor2 or fa_tensor1), null for an undefined one.
// False: not a view the operators take (rank, last stride, element type).
template <typename V, int N>
bool view_of(const Tensor& t, V* v) {
  *v = V{};
  if (!t.defined()) return true;
  if (t.dim() != N || t.stride(-1) != 1) return false;
  v->ptr = t.data_ptr();
  for (int i = 0; i < N; ++i) {
    v->sizes[i] = (uint64_t)t.size(i);
    v->strides[i] = (uint64_t)t.stride(i);
  }
  v->dtype = dtype_code(t.scalar_type());
  return v->dtype != FA_DTYPE_UNKNOWN;
}
bool view4(const Tensor& t, fa_tensor4* v) { return view_of<fa_tensor4, 4>(t, v); }
bool view2(const Tensor& t, fa_tensor2* v) { return view_of<fa_tensor2, 2>(t, v); }
// a rank-1 view has two elements or more: one element or none is a device scalar
bool view1(const Tensor& t, fa_tensor1* v) {
  return view_of<fa_tensor1, 1>(t, v) && (!t.defined() || t.numel() > 1);
}
bool view0(const Tensor& t, fa_tensor0* v) {
  *v = fa_tensor0{};
  if (!t.defined()) return true;
  if (t.dim() != 1 || t.numel() > 1) return false;
  v->ptr = t.data_ptr();
  v->dtype = dtype_code(t.scalar_type());
  return v->dtype != FA_DTYPE_UNKNOWN;
}

fa_tensor0 scalar_at(const Tensor& block, int i) {
  fa_tensor0 v{};
  v.ptr = static_cast<uint64_t*>(block.data_ptr()) + i;
  v.dtype = FA_DTYPE_UINT64;
  return v;
}

void* current_stream() { return c10::hip::getCurrentHIPStream().stream(); }

const char* error_name(int rc) {
  switch (rc) {
    case 1: return "hipErrorInvalidValue";
    case 2: return "hipErrorOutOfMemory";
    case 13: return "hipErrorInvalidSymbol";
    case 209: return "hipErrorNoBinaryForGpu";
    case 217: return "hipErrorPeerAccessUnsupported";
    case 700: return "hipErrorIllegalAddress";
    case 801: return "hipErrorNotSupported";
    default: return "hipError";
  }
}

void check_rc(int rc, bool backend_is_not_implemented) {
  if (rc == FA_SUCCESS) return;
  TORCH_CHECK_NOT_IMPLEMENTED(!(backend_is_not_implemented && rc == FA_ERROR_PEER_ACCESS_UNSUPPORTED),
                              "backend cannot take this input");
  TORCH_CHECK(false, "flash operator failed: <hipError_t.", error_name(rc), ": ", rc, ">");
}

// delta of the split backward, allocated when the library asks for it
struct LazyDelta {
  fa_lazy_tensor2 c{};
  Tensor held;
  at::IntArrayRef sizes;
  at::Device device;
  LazyDelta(at::IntArrayRef s, at::Device d) : sizes(s), device(d) {
    c.cookie = this;
    c.acquire = &acquire;
    c.dispose = &dispose;
  }
  static int acquire(fa_lazy_tensor2* self, fa_tensor2* out) {
    auto* me = static_cast<LazyDelta*>(self->cookie);
    try {
      me->held = at::empty(me->sizes, at::TensorOptions(at::kFloat).device(me->device));
      return view2(me->held, out) ? 0 : 1;
    } catch (...) {
      return 1;
    }
  }
  static void dispose(fa_lazy_tensor2* self) { static_cast<LazyDelta*>(self->cookie)->held.reset(); }
};

// Scratch memory of a forward, from torch's allocator: ordered with the stream, and a graph's own under capture.
// It is taken on the current device, whose current stream the call runs on: on another device (where the
// caller's tensors lie, say) the allocator could hand it on before the kernels are done with it.
struct Scratch {
  fa_allocator c{};
  Tensor held;
  Scratch() {
    c.cookie = this;
    c.alloc = &alloc;
  }
  static void* alloc(fa_allocator* self, uint64_t bytes) {
    auto* me = static_cast<Scratch*>(self->cookie);
    try {
      const at::Device device(at::kCUDA, c10::hip::current_device());
      me->held = at::empty({(int64_t)bytes}, at::TensorOptions(at::kByte).device(device));
      return me->held.data_ptr();
    } catch (...) {
      return nullptr;
    }
  }
};

// ---- what `attention`, the custom ops and their backwards share -----------------------------------

struct Mask { int type = 0, left = 0, right = 0; };

struct Varlen {
  Tensor cu_q, cu_k;      // undefined: dense
  int max_q = 0, max_k = 0;
};

template <typename P>
void fill_common(P& p, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& b, double scale, double dropout_p,
                 const Mask& mask, const Varlen& vl) {
  const bool ok = view4(q, &p.Q) && view4(k, &p.K) && view4(v, &p.V) &&
                  view4(b.defined() && b.numel() > 0 ? b : Tensor(), &p.B);
  TORCH_CHECK(ok, "the last stride of tensors must be 1");
  p.Sm_scale = (float)scale;
  p.dropout_p = (float)dropout_p;
  p.causal_type = (int8_t)mask.type;
  p.window_left = mask.left;
  p.window_right = mask.right;
  if (vl.cu_q.defined()) {
    TORCH_CHECK(view1(vl.cu_q, &p.cu_seqlens_q) && view1(vl.cu_k, &p.cu_seqlens_k), "no sequence");
    p.Max_seqlen_q = vl.max_q;
    p.Max_seqlen_k = vl.max_k;
    p.varlen_type = FA_VARLEN_COMPACT;
  }
}

int run_forward(fa_fwd_params& p, const Tensor& lse, const Tensor& o, const Tensor& encoded) {
  TORCH_CHECK(view2(lse, &p.L) && view4(o, &p.Out) && view4(encoded, &p.encoded_softmax), "outputs");
  Scratch scratch;
  return fa_attn_fwd_alloc(&p, FA_FWD_PARAMS_VERSION, current_stream(), nullptr, &scratch.c);
}

int run_backward(fa_bwd_params& p, const Tensor& o, const Tensor& dout, const Tensor& lse, const Tensor& dq,
                 const Tensor& dk, const Tensor& dv, const Tensor& db, int backend) {
  const Tensor d = dout.stride(-1) == 1 ? dout : dout.contiguous();
  TORCH_CHECK(view4(o, &p.Out) && view4(d, &p.DO) && view2(lse, &p.L) && view4(dq, &p.DQ) && view4(dk, &p.DK) &&
                  view4(dv, &p.DV) && view4(db, &p.DB), "the last stride of tensors must be 1");
  LazyDelta delta(lse.sizes(), lse.device());
  p.D = delta.c;
  fa_options opt{backend, 0};
  return fa_attn_bwd(&p, FA_BWD_PARAMS_VERSION, current_stream(), backend >= 0 ? &opt : nullptr);
}

// `n` 32-bit words of the host in a new device tensor, without a copy or a synchronisation: they
// travel as kernel arguments.  Beyond a thousand words one copy is cheaper.
Tensor words_on_device(const std::vector<uint32_t>& words, at::ScalarType type, int64_t numel, at::Device device) {
  if (words.size() > 1024) {
    Tensor host = at::empty({numel}, at::TensorOptions(type));
    memcpy(host.data_ptr(), words.data(), words.size() * 4);
    return host.to(device);
  }
  Tensor t = at::empty({numel}, at::TensorOptions(type).device(device));
  check_rc(fa_write_words(t.data_ptr(), words.data(), (int32_t)words.size(), current_stream()), false);
  return t;
}

void push64(std::vector<uint32_t>& w, uint64_t x) {
  w.push_back((uint32_t)x);
  w.push_back((uint32_t)(x >> 32));
}

// ---- autograd.attention / attention_varlen -----------------------------------------------------------

struct AttentionOptions {
  Mask mask;
  double scale = 0, dropout_p = 0;
  bool encoded = false, lse = false, fillnan = false;
  int backend = -1;
  uint64_t seed = 0, offset1 = 0, offset2 = 0;
  Varlen vl;
  int64_t num_seqlens = 0;
};

struct AttentionResult { Tensor o, lse, encoded, philox; };

AttentionResult attention_forward(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& b,
                                  const AttentionOptions& x) {
  AttentionResult r;
  const c10::DeviceGuard guard(q.device());
  fa_fwd_params p{};
  fill_common(p, q, k, v, b, x.scale, x.dropout_p, x.mask, x.vl);
  const bool packed = x.vl.cu_q.defined();
  r.o = at::empty({q.size(0), q.size(1), q.size(2), v.size(3)}, q.options());
  r.lse = at::empty({packed ? q.size(1) : q.size(0) * q.size(1), q.size(2)}, q.options().dtype(at::kFloat));
  if (x.fillnan) {
    r.o.fill_(std::numeric_limits<double>::quiet_NaN());
    r.lse.fill_(std::numeric_limits<double>::quiet_NaN());
  }
  if (x.encoded)
    r.encoded = packed ? at::zeros({x.num_seqlens, q.size(1), x.vl.max_q, x.vl.max_k}, q.options())
                       : at::zeros({q.size(0), q.size(1), q.size(2), k.size(2)}, q.options());
  if (x.dropout_p > 0) {
    // seed and offset of this call, and where the kernel writes those that the backward uses
    std::vector<uint32_t> w;
    push64(w, x.seed); push64(w, x.offset1); push64(w, 0); push64(w, 0);
    r.philox = words_on_device(w, at::kLong, 4, q.device());
    p.philox_seed_ptr = scalar_at(r.philox, 0);
    p.philox_offset1 = scalar_at(r.philox, 1);
    p.philox_offset2 = x.offset2;
    p.philox_seed_output = scalar_at(r.philox, 2);
    p.philox_offset_output = scalar_at(r.philox, 3);
  }
  check_rc(run_forward(p, r.lse, r.o, r.encoded), true);
  return r;
}

struct AttentionFunction : torch::autograd::Function<AttentionFunction> {
  static variable_list forward(AutogradContext* ctx, const Tensor& q, const Tensor& k, const Tensor& v,
                               const std::optional<Tensor>& b, const AttentionOptions* x) {
    AttentionResult r = attention_forward(q, k, v, b.value_or(Tensor()), *x);
    ctx->save_for_backward({q, k, v, b.value_or(Tensor()), r.o, r.lse, r.philox, x->vl.cu_q, x->vl.cu_k});
    ctx->set_materialize_grads(false);
    auto& d = ctx->saved_data;
    d["mask"] = c10::IntArrayRef({x->mask.type, x->mask.left, x->mask.right, x->backend, x->vl.max_q, x->vl.max_k});
    d["scale"] = x->scale;
    d["dropout_p"] = x->dropout_p;
    // (an undefined tensor cannot be an output of a Function)
    variable_list out{r.o};
    if (x->encoded) out.push_back(r.encoded);
    if (x->lse) out.push_back(r.lse);
    return out;
  }

  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const variable_list s = ctx->get_saved_variables();
    const Tensor &q = s[0], &k = s[1], &v = s[2], &b = s[3];
    const std::vector<int64_t> ints = ctx->saved_data["mask"].toIntVector();
    const c10::DeviceGuard guard(q.device());
    fa_bwd_params p{};
    const double dropout_p = ctx->saved_data["dropout_p"].toDouble();
    fill_common(p, q, k, v, b, ctx->saved_data["scale"].toDouble(), dropout_p,
                Mask{(int)ints[0], (int)ints[1], (int)ints[2]}, Varlen{s[7], s[8], (int)ints[4], (int)ints[5]});
    if (dropout_p > 0) {
      p.philox_seed_ptr = scalar_at(s[6], 2);
      p.philox_offset1 = scalar_at(s[6], 3);
    }
    const Tensor dout = grads[0].defined() ? grads[0] : at::zeros_like(s[4]);
    const Tensor dq = at::empty_like(q), dk = at::empty_like(k), dv = at::empty_like(v);
    const Tensor db = b.defined() && ctx->needs_input_grad(3) ? at::empty_like(b) : Tensor();
    check_rc(run_backward(p, s[4], dout, s[5], dq, dk, dv, db, (int)ints[3]), true);
    return {dq, dk, dv, db, Tensor()};
  }
};

// There is no forward-mode formula.  A call without a gradient goes past the Function, whose own error would
// come after the launch: without this check such a call would answer without the tangent.
void refuse_tangents(std::initializer_list<const Tensor*> inputs) {
  if (torch::autograd::ForwardADLevel::try_get_by_idx(0) == nullptr) return;      // (the tensors' own look takes locks)
  for (const Tensor* t : inputs)
    TORCH_CHECK_NOT_IMPLEMENTED(!t->defined() || !t->_fw_grad(0).defined(),
                                "forward-mode AD of the attention operators (jvp) is not implemented");
}

// (Out, encoded softmax, logsumexp); the last two undefined unless asked for
variable_list attention(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& b, const AttentionOptions& x) {
  refuse_tangents({&q, &k, &v, &b});
  const bool grad = at::GradMode::is_enabled() && (q.requires_grad() || k.requires_grad() || v.requires_grad() ||
                                                   (b.defined() && b.requires_grad()));
  if (grad) {
    const variable_list r = AttentionFunction::apply(q, k, v, b.defined() ? std::optional<Tensor>(b) : std::nullopt, &x);
    return {r[0], x.encoded ? r[1] : Tensor(), x.lse ? r.back() : Tensor()};
  }
  at::AutoDispatchBelowADInplaceOrView below;
  AttentionResult r = attention_forward(q, k, v, b, x);
  return {r.o, r.encoded, x.lse ? r.lse : Tensor()};
}

// ---- torch.ops.aotriton_amd.* -------------------------------------------------------------------------

using FwdSig = std::tuple<Tensor, Tensor>(const Tensor&, const Tensor&, const Tensor&, const std::optional<Tensor>&,
                                          double, c10::SymInt, c10::SymInt, c10::SymInt, double, const Tensor&,
                                          const Tensor&);
using BwdSig = std::tuple<Tensor, Tensor, Tensor, Tensor>(
    const Tensor&, const Tensor&, const Tensor&, const Tensor&, const std::optional<Tensor>&, const Tensor&,
    const Tensor&, double, c10::SymInt, c10::SymInt, c10::SymInt, double, const Tensor&, const Tensor&, bool,
    c10::SymInt);

const c10::TypedOperatorHandle<FwdSig>& forward_op() {
  static const auto op = c10::Dispatcher::singleton()
                             .findSchemaOrThrow("aotriton_amd::flash_attention_forward", "").typed<FwdSig>();
  return op;
}
// flash_attention_forward_key_mask(q, k, v, mask, sm_scale): a boolean mask that is the same for all query rows, 4-D and
// broadcast here
using MaskSig = std::tuple<Tensor, Tensor>(const Tensor&, const Tensor&, const Tensor&, const Tensor&, double);
const c10::TypedOperatorHandle<MaskSig>& key_mask_op() {
  static const auto op = c10::Dispatcher::singleton()
                             .findSchemaOrThrow("aotriton_amd::flash_attention_forward_key_mask", "").typed<MaskSig>();
  return op;
}
const c10::TypedOperatorHandle<BwdSig>& backward_op() {
  static const auto op = c10::Dispatcher::singleton()
                             .findSchemaOrThrow("aotriton_amd::flash_attention_backward", "").typed<BwdSig>();
  return op;
}

void set_philox(fa_tensor0* seed, fa_tensor0* offset, const Tensor& s, const Tensor& o) {
  TORCH_CHECK(view0(s, seed) && view0(o, offset), "philox seed and offset are one-element tensors");
}

std::tuple<Tensor, Tensor> forward_kernel(const Tensor& q, const Tensor& k, const Tensor& v,
                                          const std::optional<Tensor>& bias, double dropout_p, int64_t causal_type,
                                          int64_t window_left, int64_t window_right, double sm_scale,
                                          const Tensor& seed, const Tensor& offset) {
  const c10::DeviceGuard guard(q.device());
  fa_fwd_params p{};
  fill_common(p, q, k, v, bias.value_or(Tensor()), sm_scale, dropout_p,
              Mask{(int)causal_type, (int)window_left, (int)window_right}, Varlen{});
  if (dropout_p > 0) set_philox(&p.philox_seed_ptr, &p.philox_offset1, seed, offset);
  Tensor o = at::empty({q.size(0), q.size(1), q.size(2), v.size(3)}, q.options());
  Tensor lse = at::empty({q.size(0) * q.size(1), q.size(2)}, q.options().dtype(at::kFloat));
  check_rc(run_forward(p, lse, o, Tensor()), false);
  return {std::move(o), std::move(lse)};
}

// log(1) = 0 where the key is visible, log(0) = -inf where it is not: the additive mask in one kernel
Tensor additive_mask(const Tensor& mask, const at::TensorOptions& like) {
  Tensor additive = at::empty_like(mask, like);
  at::log_out(additive, mask);
  return additive;
}
Tensor unit_stride(const Tensor& t) { return t.stride(-1) == 1 ? t : t.contiguous(); }
Tensor broadcast_bias(const Tensor& m, const Tensor& q, const Tensor& k) {
  return unit_stride(m.expand({q.size(0), q.size(1), q.size(2), k.size(2)}));
}
std::tuple<Tensor, Tensor> forward_additive(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& mask, double sm_scale) {
  const Tensor none = at::empty({0}, q.options().dtype(at::kUInt64));      // not read
  return forward_op().call(q, k, v, std::optional<Tensor>(broadcast_bias(additive_mask(mask, q.options()), q, k)), 0.0, FA_CAUSAL_NONE, 0, 0,
                           sm_scale, none, none);
}

std::tuple<Tensor, Tensor> key_mask_kernel(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& mask, double sm_scale) {
  TORCH_CHECK(mask.scalar_type() == at::kBool && mask.dim() == 4 && mask.size(2) == 1 && mask.device() == q.device(),
              "a boolean (.., .., 1, keys) mask on the device of the queries");
  const c10::DeviceGuard guard(q.device());
  fa_fwd_params p{};
  fill_common(p, q, k, v, Tensor(), sm_scale, 0.0, Mask{}, Varlen{});
  const Tensor m = mask.expand({q.size(0), q.size(1), 1, k.size(2)});
  Tensor o = at::empty({q.size(0), q.size(1), q.size(2), v.size(3)}, q.options());
  Tensor lse = at::empty({q.size(0) * q.size(1), q.size(2)}, q.options().dtype(at::kFloat));
  int rc = FA_ERROR_NOT_SUPPORTED;
  // (what is known here to be refused is not asked for)
  if (m.numel() > 0 && q.element_size() == 2 && q.size(3) <= 128 && v.size(3) <= 128) {
    p.B.ptr = m.data_ptr();
    for (int i = 0; i < 4; ++i) {
      p.B.sizes[i] = (uint64_t)(i == 2 ? q.size(2) : m.size(i));
      p.B.strides[i] = (uint64_t)(i == 2 ? 0 : m.stride(i));
    }
    p.B.dtype = FA_DTYPE_UINT8;
    TORCH_CHECK(view2(lse, &p.L) && view4(o, &p.Out), "outputs");
    Scratch scratch;
    rc = fa_attn_fwd_key_mask(&p, FA_FWD_PARAMS_VERSION, current_stream(), nullptr, &scratch.c);
  }
  if (rc == FA_ERROR_NOT_SUPPORTED) {      // nothing was launched: the additive mask instead, into the same outputs
    const Tensor b = broadcast_bias(additive_mask(mask, q.options()), q, k);
    TORCH_CHECK(view4(b.numel() > 0 ? b : Tensor(), &p.B), "the last stride of tensors must be 1");
    rc = run_forward(p, lse, o, Tensor());
  }
  check_rc(rc, false);
  return {std::move(o), std::move(lse)};
}

std::tuple<Tensor, Tensor, Tensor, Tensor> backward_kernel(
    const Tensor& dout, const Tensor& q, const Tensor& k, const Tensor& v, const std::optional<Tensor>& bias,
    const Tensor& out, const Tensor& lse, double dropout_p, int64_t causal_type, int64_t window_left,
    int64_t window_right, double sm_scale, const Tensor& seed, const Tensor& offset, bool need_dbias, int64_t backend) {
  const c10::DeviceGuard guard(q.device());
  fa_bwd_params p{};
  fill_common(p, q, k, v, bias.value_or(Tensor()), sm_scale, dropout_p,
              Mask{(int)causal_type, (int)window_left, (int)window_right}, Varlen{});
  if (dropout_p > 0) set_philox(&p.philox_seed_ptr, &p.philox_offset1, seed, offset);
  const bool want_db = need_dbias && bias.has_value() && bias->defined();
  Tensor dq = at::empty(q.sizes(), q.options()), dk = at::empty(k.sizes(), q.options()),
         dv = at::empty(v.sizes(), q.options());
  Tensor db = want_db ? at::empty(bias->sizes(), q.options()) : at::empty({0}, q.options());
  check_rc(run_backward(p, out, dout, lse, dq, dk, dv, want_db ? db : Tensor(), (int)backend), false);
  return {std::move(dq), std::move(dk), std::move(dv), std::move(db)};
}

std::tuple<Tensor, Tensor> philox_kernel(const Tensor& like, int64_t increment) {
  const c10::DeviceGuard guard(like.device());
  at::Generator gen = at::globalContext().defaultGenerator(like.device());
  uint64_t seed, offset;
  {
    std::lock_guard<std::mutex> lock(gen.mutex());
    seed = gen.current_seed();
    offset = gen.get_offset();
    gen.set_offset(offset + (uint64_t)((increment + 3) / 4 * 4));
  }
  std::vector<uint32_t> w;
  push64(w, seed);
  const Tensor s = words_on_device(w, at::kLong, 1, like.device());
  w.clear();
  push64(w, offset);
  const Tensor o = words_on_device(w, at::kLong, 1, like.device());
  return {s.view(at::kUInt64), o.view(at::kUInt64)};
}

struct OpFunction : torch::autograd::Function<OpFunction> {
  static variable_list forward(AutogradContext* ctx, const Tensor& q, const Tensor& k, const Tensor& v,
                               const std::optional<Tensor>& bias, double dropout_p, const c10::SymInt& causal_type,
                               const c10::SymInt& window_left, const c10::SymInt& window_right, double sm_scale,
                               const Tensor& seed, const Tensor& offset) {
    at::AutoDispatchBelowADInplaceOrView below;
    auto [o, lse] = forward_op().call(q, k, v, bias, dropout_p, causal_type, window_left, window_right, sm_scale, seed, offset);
    ctx->save_for_backward({q, k, v, bias.value_or(Tensor()), o, lse, seed, offset});
    ctx->set_materialize_grads(false);
    auto& d = ctx->saved_data;
    d["dropout_p"] = dropout_p;
    d["sm_scale"] = sm_scale;
    d["type"] = causal_type;
    d["left"] = window_left;
    d["right"] = window_right;
    return {o, lse};
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const variable_list s = ctx->get_saved_variables();
    auto& d = ctx->saved_data;
    const Tensor& b = s[3];
    const bool need_dbias = b.defined() && ctx->needs_input_grad(3);
    const Tensor dout = grads[0].defined() ? grads[0] : at::zeros_like(s[4]);
    auto [dq, dk, dv, db] = backward_op().call(dout, s[0], s[1], s[2], b.defined() ? std::optional<Tensor>(b) : std::nullopt,
                                               s[4], s[5], d["dropout_p"].toDouble(), d["type"].toSymInt(), d["left"].toSymInt(),
                                               d["right"].toSymInt(), d["sm_scale"].toDouble(), s[6], s[7], need_dbias, -1);
    return {dq, dk, dv, need_dbias ? db : Tensor(), Tensor(), Tensor(), Tensor(), Tensor(), Tensor(), Tensor(), Tensor()};
  }
};

std::tuple<Tensor, Tensor> forward_autograd(const Tensor& q, const Tensor& k, const Tensor& v,
                                            const std::optional<Tensor>& bias, double dropout_p, c10::SymInt causal_type,
                                            c10::SymInt window_left, c10::SymInt window_right, double sm_scale,
                                            const Tensor& seed, const Tensor& offset) {
  const bool grad = at::GradMode::is_enabled() && (q.requires_grad() || k.requires_grad() || v.requires_grad() ||
                                                   (bias.has_value() && bias->defined() && bias->requires_grad()));
  if (!grad) {
    at::AutoDispatchBelowADInplaceOrView below;
    return forward_op().call(q, k, v, bias, dropout_p, causal_type, window_left, window_right, sm_scale, seed, offset);
  }
  const Tensor b = bias.value_or(Tensor());
  refuse_tangents({&q, &k, &v, &b});
  variable_list r = OpFunction::apply(q, k, v, bias, dropout_p, causal_type, window_left, window_right, sm_scale, seed, offset);
  return {r[0], r[1]};
}

std::tuple<Tensor, Tensor> key_mask_autograd(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& mask, double sm_scale) {
  if (at::GradMode::is_enabled() && (q.requires_grad() || k.requires_grad() || v.requires_grad()))
    return forward_additive(q, k, v, mask, sm_scale);      // (the backward takes an additive mask)
  at::AutoDispatchBelowADInplaceOrView below;
  return key_mask_op().call(q, k, v, mask, sm_scale);
}

// The backward op has no derivative of its own.  Its results say so when something asks for one; without
// an Autograd kernel PyTorch would hand back undefined gradients with a warning, and a double backward
// through flash_attention_forward would run this op on zeros.
struct OpBackwardFunction : torch::autograd::Function<OpBackwardFunction> {
  static variable_list forward(AutogradContext*, const Tensor& dout, const Tensor& q, const Tensor& k, const Tensor& v,
                               const std::optional<Tensor>& bias, const Tensor& out, const Tensor& lse, double dropout_p,
                               const c10::SymInt& causal_type, const c10::SymInt& window_left,
                               const c10::SymInt& window_right, double sm_scale, const Tensor& seed,
                               const Tensor& offset, bool need_dbias, const c10::SymInt& backend) {
    at::AutoDispatchBelowADInplaceOrView below;
    auto [dq, dk, dv, db] = backward_op().call(dout, q, k, v, bias, out, lse, dropout_p, causal_type, window_left,
                                               window_right, sm_scale, seed, offset, need_dbias, backend);
    return {dq, dk, dv, db};
  }
  static variable_list backward(AutogradContext*, variable_list) {
    TORCH_CHECK(false, "Trying to backward through aotriton_amd::flash_attention_backward, which has no autograd formula: "
                       "second derivatives of the attention operators are not implemented");
  }
};

std::tuple<Tensor, Tensor, Tensor, Tensor> backward_autograd(
    const Tensor& dout, const Tensor& q, const Tensor& k, const Tensor& v, const std::optional<Tensor>& bias,
    const Tensor& out, const Tensor& lse, double dropout_p, c10::SymInt causal_type, c10::SymInt window_left,
    c10::SymInt window_right, double sm_scale, const Tensor& seed, const Tensor& offset, bool need_dbias,
    c10::SymInt backend) {
  const bool grad = at::GradMode::is_enabled() &&
                    (dout.requires_grad() || q.requires_grad() || k.requires_grad() || v.requires_grad() ||
                     (bias.has_value() && bias->defined() && bias->requires_grad()) || out.requires_grad() ||
                     lse.requires_grad());
  if (!grad) {
    at::AutoDispatchBelowADInplaceOrView below;
    return backward_op().call(dout, q, k, v, bias, out, lse, dropout_p, causal_type, window_left, window_right, sm_scale,
                              seed, offset, need_dbias, backend);
  }
  const Tensor b = bias.value_or(Tensor());
  refuse_tangents({&dout, &q, &k, &v, &b, &out, &lse});
  variable_list r = OpBackwardFunction::apply(dout, q, k, v, bias, out, lse, dropout_p, causal_type, window_left, window_right,
                                              sm_scale, seed, offset, need_dbias, backend);
  return {r[0], r[1], r[2], r[3]};
}

// (pt2_compliant_tag: fake implementations and Autograd kernels are there, so that torch.compile may keep the
// ops in its graphs also where it is told to take compliant ops only)
TORCH_LIBRARY(aotriton_amd, m) {
  const std::vector<at::Tag> compliant{at::Tag::pt2_compliant_tag};
  m.def("philox_state(Tensor like, SymInt increment) -> (Tensor, Tensor)",
        {at::Tag::pt2_compliant_tag, at::Tag::nondeterministic_seeded});
  m.def("flash_attention_forward(Tensor q, Tensor k, Tensor v, Tensor? bias, float dropout_p, SymInt causal_type, "
        "SymInt window_left, SymInt window_right, float sm_scale, Tensor philox_seed, Tensor philox_offset) -> (Tensor, Tensor)",
        compliant);
  m.def("flash_attention_forward_key_mask(Tensor q, Tensor k, Tensor v, Tensor mask, float sm_scale) -> (Tensor, Tensor)", compliant);
  m.def("flash_attention_backward(Tensor dout, Tensor q, Tensor k, Tensor v, Tensor? bias, Tensor out, Tensor lse, "
        "float dropout_p, SymInt causal_type, SymInt window_left, SymInt window_right, float sm_scale, "
        "Tensor philox_seed, Tensor philox_offset, bool need_dbias, SymInt backend) -> (Tensor, Tensor, Tensor, Tensor)",
        compliant);
}
TORCH_LIBRARY_IMPL(aotriton_amd, CUDA, m) {
  m.impl("philox_state", &philox_kernel);
  m.impl("flash_attention_forward", &forward_kernel);
  m.impl("flash_attention_forward_key_mask", &key_mask_kernel);
  m.impl("flash_attention_backward", &backward_kernel);
}
TORCH_LIBRARY_IMPL(aotriton_amd, Autograd, m) {
  m.impl("flash_attention_forward", &forward_autograd);
  m.impl("flash_attention_forward_key_mask", &key_mask_autograd);
  m.impl("flash_attention_backward", &backward_autograd);
}

// ---- argument parsing of the Python functions ---------------------------------------------------------

// Reads positional arguments in order.  `odd` is set where an argument is not of the kind that the
// native path takes; the Python layer then goes through its views, which also report the error.
struct Args {
  PyObject* const* a;
  Py_ssize_t n, i = 0;
  bool odd = false;
  PyObject* next() { TORCH_CHECK(i < n, "too few arguments"); return a[i++]; }
  Tensor tensor(bool may_be_none) {
    PyObject* o = next();
    if (o == Py_None) { odd |= !may_be_none; return Tensor(); }
    if (!THPVariable_Check(o)) { odd = true; return Tensor(); }
    return THPVariable_Unpack(o);
  }
  double real() {
    const double x = PyFloat_AsDouble(next());
    if (x == -1.0 && PyErr_Occurred()) throw python_error();
    return x;
  }
  int64_t integer() {
    const long long x = PyLong_AsLongLong(next());
    if (x == -1 && PyErr_Occurred()) throw python_error();
    return x;
  }
  uint64_t word64() {
    const unsigned long long x = PyLong_AsUnsignedLongLongMask(next());
    if (x == (unsigned long long)-1 && PyErr_Occurred()) throw python_error();
    return x;
  }
  bool flag() {
    const int x = PyObject_IsTrue(next());
    if (x < 0) throw python_error();
    return x == 1;
  }
};

// attn_fwd(q, k, v, b, sm_scale, M, o, dropout_p, seed, offset1, offset2, seed_out, offset_out, encoded, type, left,
//          right, counter, cu_q, cu_k, max_q, max_k, strides_q, strides_k, varlen_type, backend, deterministic, stream)
// stream: -1 = torch's current one.  hipError_t, or None where the arguments are not plain tensors.
PyObject* py_attn_fwd(PyObject*, PyObject* const* argv, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Args a{argv, n};
  fa_fwd_params p{};
  bool ok = view4(a.tensor(false), &p.Q) && view4(a.tensor(false), &p.K) && view4(a.tensor(false), &p.V);
  if (!ok || a.odd) Py_RETURN_NONE;
  const Tensor b = a.tensor(true);
  ok = view4(b.defined() && b.numel() > 0 ? b : Tensor(), &p.B);
  p.Sm_scale = (float)a.real();
  ok &= view2(a.tensor(true), &p.L);
  const Tensor o = a.tensor(false);
  ok &= view4(o, &p.Out);
  p.dropout_p = (float)a.real();
  ok &= view0(a.tensor(false), &p.philox_seed_ptr);
  ok &= view0(a.tensor(false), &p.philox_offset1);
  p.philox_offset2 = a.word64();
  ok &= view0(a.tensor(false), &p.philox_seed_output);
  ok &= view0(a.tensor(false), &p.philox_offset_output);
  ok &= view4(a.tensor(true), &p.encoded_softmax);
  p.causal_type = (int8_t)a.integer();
  p.window_left = (int32_t)a.integer();
  p.window_right = (int32_t)a.integer();
  ok &= view0(a.tensor(false), &p.persistent_atomic_counter);
  ok &= view1(a.tensor(true), &p.cu_seqlens_q);
  ok &= view1(a.tensor(true), &p.cu_seqlens_k);
  p.Max_seqlen_q = (int32_t)a.integer();
  p.Max_seqlen_k = (int32_t)a.integer();
  ok &= view1(a.tensor(true), &p.seq_strides_q);
  ok &= view1(a.tensor(true), &p.seq_strides_k);
  p.varlen_type = (int8_t)a.integer();
  fa_options opt{};
  opt.force_backend_index = (int32_t)a.integer();
  opt.deterministic = a.flag() ? 1 : 0;
  const int64_t stream = a.integer();
  if (!ok || a.odd) Py_RETURN_NONE;
  int rc;
  {
    pybind11::gil_scoped_release no_gil;
    // torch's allocator orders its memory with torch's current stream only
    Scratch scratch;
    rc = stream == -1 ? fa_attn_fwd_alloc(&p, FA_FWD_PARAMS_VERSION, current_stream(), &opt, &scratch.c)
                      : fa_attn_fwd(&p, FA_FWD_PARAMS_VERSION, reinterpret_cast<void*>(stream), &opt);
  }
  return PyLong_FromLong(rc);
  END_HANDLE_TH_ERRORS
}

// attn_bwd(q, k, v, b, sm_scale, o, dout, dq, dk, dv, db, L, delta, lazy_delta, dropout_p, seed, offset1, offset2, type,
//          left, right, cu_q, cu_k, max_q, max_k, strides_q, strides_k, varlen_type, backend, deterministic, stream)
// lazy_delta: delta is allocated here when the library asks for it.
PyObject* py_attn_bwd(PyObject*, PyObject* const* argv, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Args a{argv, n};
  fa_bwd_params p{};
  bool ok = view4(a.tensor(false), &p.Q) && view4(a.tensor(false), &p.K) && view4(a.tensor(false), &p.V);
  if (!ok || a.odd) Py_RETURN_NONE;
  const Tensor b = a.tensor(true);
  ok = view4(b.defined() && b.numel() > 0 ? b : Tensor(), &p.B);
  p.Sm_scale = (float)a.real();
  ok &= view4(a.tensor(false), &p.Out);
  ok &= view4(a.tensor(false), &p.DO);
  ok &= view4(a.tensor(false), &p.DQ);
  ok &= view4(a.tensor(false), &p.DK);
  ok &= view4(a.tensor(false), &p.DV);
  ok &= view4(a.tensor(true), &p.DB);
  const Tensor lse = a.tensor(false);
  ok &= view2(lse, &p.L);
  const Tensor delta = a.tensor(true);
  ok &= view2(delta, &p.D.eager);
  const bool lazy = a.flag();
  p.dropout_p = (float)a.real();
  ok &= view0(a.tensor(false), &p.philox_seed_ptr);
  ok &= view0(a.tensor(false), &p.philox_offset1);
  p.philox_offset2 = a.word64();
  p.causal_type = (int8_t)a.integer();
  p.window_left = (int32_t)a.integer();
  p.window_right = (int32_t)a.integer();
  ok &= view1(a.tensor(true), &p.cu_seqlens_q);
  ok &= view1(a.tensor(true), &p.cu_seqlens_k);
  p.Max_seqlen_q = (int32_t)a.integer();
  p.Max_seqlen_k = (int32_t)a.integer();
  ok &= view1(a.tensor(true), &p.seq_strides_q);
  ok &= view1(a.tensor(true), &p.seq_strides_k);
  p.varlen_type = (int8_t)a.integer();
  fa_options opt{};
  opt.force_backend_index = (int32_t)a.integer();
  opt.deterministic = a.flag() ? 1 : 0;
  const int64_t stream = a.integer();
  if (!ok || a.odd) Py_RETURN_NONE;
  LazyDelta own(lse.sizes(), lse.device());
  if (lazy) p.D = own.c;
  int rc;
  {
    pybind11::gil_scoped_release no_gil;
    rc = fa_attn_bwd(&p, FA_BWD_PARAMS_VERSION, stream == -1 ? current_stream() : reinterpret_cast<void*>(stream), &opt);
  }
  return PyLong_FromLong(rc);
  END_HANDLE_TH_ERRORS
}

PyObject* wrap(const Tensor& t) {
  if (!t.defined()) Py_RETURN_NONE;
  return THPVariable_Wrap(t);
}

AttentionOptions read_options(Args& a) {
  AttentionOptions x;
  x.mask.type = (int)a.integer();
  x.mask.left = (int)a.integer();
  x.mask.right = (int)a.integer();
  x.scale = a.real();
  x.dropout_p = a.real();
  x.encoded = a.flag();
  x.lse = a.flag();
  x.fillnan = a.flag();
  x.backend = (int)a.integer();
  x.seed = a.word64();
  x.offset1 = a.word64();
  x.offset2 = a.word64();
  return x;
}

PyObject* pack_result(const variable_list& r) {
  PyObject* t = PyTuple_New(3);
  if (t == nullptr) throw python_error();
  for (int i = 0; i < 3; ++i) PyTuple_SET_ITEM(t, i, wrap(i < (int)r.size() ? r[i] : Tensor()));
  return t;
}

// attention(q, k, v, b, type, left, right, sm_scale, dropout_p, encoded, lse, fillnan, backend, seed, offset1, offset2)
PyObject* py_attention(PyObject*, PyObject* const* argv, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Args a{argv, n};
  const Tensor q = a.tensor(false), k = a.tensor(false), v = a.tensor(false), b = a.tensor(true);
  TORCH_CHECK_TYPE(!a.odd, "q, k, v and the bias are tensors");
  AttentionOptions x = read_options(a);
  variable_list r;
  {
    pybind11::gil_scoped_release no_gil;
    r = attention(q, k, v, b, x);
  }
  return pack_result(r);
  END_HANDLE_TH_ERRORS
}

std::vector<int64_t> int_list(PyObject* o) {
  TORCH_CHECK_TYPE(PyList_Check(o), "a list of lengths");
  std::vector<int64_t> v((size_t)PyList_GET_SIZE(o));
  for (size_t i = 0; i < v.size(); ++i) {
    v[i] = PyLong_AsLongLong(PyList_GET_ITEM(o, (Py_ssize_t)i));
    if (v[i] == -1 && PyErr_Occurred()) throw python_error();
  }
  return v;
}

// Appends the offsets of sequences of these lengths in a packed (1, H, tokens, D) tensor and returns the
// longest length.  The lengths have to add up to the tokens: rows past them would be left unwritten (Out, logsumexp,
// gradients), and with more the kernels would run past the tensors.
int64_t push_offsets(std::vector<uint32_t>* words, const std::vector<int64_t>& lens, const Tensor& packed, const char* side) {
  TORCH_CHECK_VALUE(packed.dim() == 4, "packed sequences are (1, heads, tokens, head_dim) tensors");
  TORCH_CHECK_VALUE(!lens.empty(), "no ", side, " sequence");
  const int64_t tokens = packed.size(2);
  TORCH_CHECK_VALUE(tokens <= std::numeric_limits<int32_t>::max(), "offsets of packed sequences are 32-bit");
  int64_t sum = 0, longest = 0;
  words->push_back(0);
  for (const int64_t len : lens) {
    TORCH_CHECK_VALUE(len >= 0 && len <= tokens - sum, side, " sequence lengths must not be negative and must add up to the ",
                      tokens, " packed tokens");
    sum += len;
    longest = std::max(longest, len);
    words->push_back((uint32_t)sum);
  }
  TORCH_CHECK_VALUE(sum == tokens, side, " sequence lengths add up to ", sum, ", the packed tensor holds ", tokens, " tokens");
  return longest;
}

// attention_varlen(q, k, v, lens_q, lens_k, then as attention from `type` on): compact packed sequences
PyObject* py_attention_varlen(PyObject*, PyObject* const* argv, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Args a{argv, n};
  const Tensor q = a.tensor(false), k = a.tensor(false), v = a.tensor(false);
  TORCH_CHECK_TYPE(!a.odd, "q, k and v are tensors");
  const std::vector<int64_t> lq = int_list(a.next()), lk = int_list(a.next());
  AttentionOptions x = read_options(a);
  variable_list r;
  refuse_tangents({&q, &k, &v});
  {
    pybind11::gil_scoped_release no_gil;
    std::vector<uint32_t> w;
    w.reserve(lq.size() + lk.size() + 2);
    const int64_t longest[2] = {push_offsets(&w, lq, q, "query"), push_offsets(&w, lk, k, "key")};
    const c10::DeviceGuard guard(q.device());
    at::AutoDispatchBelowADInplaceOrView below;
    const Tensor cu = words_on_device(w, at::kInt, (int64_t)w.size(), q.device());
    x.vl.cu_q = cu.narrow(0, 0, (int64_t)lq.size() + 1);
    x.vl.cu_k = cu.narrow(0, (int64_t)lq.size() + 1, (int64_t)lk.size() + 1);
    x.vl.max_q = (int)longest[0];
    x.vl.max_k = (int)longest[1];
    x.num_seqlens = (int64_t)lq.size();
  }
  {
    pybind11::gil_scoped_release no_gil;
    r = attention(q, k, v, Tensor(), x);
  }
  return pack_result(r);
  END_HANDLE_TH_ERRORS
}

// ---- F.scaled_dot_product_attention-shaped ----------------------------------------------------------------

struct Sdpa {
  Tensor q, k, v, bias;
  Tensor key_mask;      // instead of the bias: a boolean mask of one row, 4-D, not broadcast yet
  double scale = 0;
};

// sdpa.py's prepare(): argument checks, unit last strides, the mask as an additive (B, H, L, S) bias
Sdpa prepare(const Tensor& query, const Tensor& key, const Tensor& value, const Tensor& mask, bool is_causal,
             std::optional<double> scale, bool gqa, bool take_key_mask = false) {
  TORCH_CHECK_VALUE(query.dim() == 4 && key.dim() == 4 && value.dim() == 4, "expected (batch, heads, seq, head_dim) tensors");
  TORCH_CHECK_VALUE(!(is_causal && mask.defined()), "attn_mask and is_causal cannot both be set");
  const int64_t hq = query.size(1), hk = key.size(1);
  TORCH_CHECK_VALUE(hq == hk || (gqa && hk > 0 && hq % hk == 0 && value.size(1) == hk),
                    "number of heads of query and key/value differ; pass enable_gqa=True for grouped queries");
  Sdpa s;
  s.scale = scale.has_value() ? *scale : 1.0 / std::sqrt((double)query.size(-1));
  s.q = unit_stride(query);
  s.k = unit_stride(key);
  s.v = unit_stride(value);
  if (mask.defined()) {
    Tensor m = mask;
    if (m.scalar_type() == at::kBool) {
      if (take_key_mask && m.dim() > 0 && m.dim() <= 4 && (m.dim() == 1 || m.size(-2) == 1) && m.size(-1) == s.k.size(2) &&
          m.device() == s.q.device()) {
        while (m.dim() < 4) m = m.unsqueeze(0);
        s.key_mask = m;
        return s;
      }
      m = additive_mask(m, s.q.options());
    } else if (m.scalar_type() != s.q.scalar_type()) {
      m = m.to(s.q.scalar_type());
    }
    while (m.dim() < 4) m = m.unsqueeze(0);
    s.bias = broadcast_bias(m, s.q, s.k);
  }
  return s;
}

// Tracers (make_fx, AOTAutograd) and other dispatch modes, tensors that dispatch to Python, functorch transforms: sizes
// may be symbols there, and reading them here as integers would fix them in the trace.  The Python route keeps them.
bool traced(std::initializer_list<const Tensor*> inputs) {
  static constexpr c10::DispatchKeySet keys({c10::DispatchKey::Python, c10::DispatchKey::FuncTorchBatched,
                                             c10::DispatchKey::FuncTorchGradWrapper});
  if (c10::impl::TorchDispatchModeTLS::any_modes_set()) return true;
  for (const Tensor* t : inputs)
    if (t->defined() && t->key_set().has_any(keys)) return true;
  return false;
}

struct SdpaArgs {
  Tensor q, k, v, mask;
  double dropout_p;
  bool causal;
  std::optional<double> scale;
  bool gqa;
};

SdpaArgs read_sdpa(Args& a) {
  SdpaArgs s;
  s.q = a.tensor(false); s.k = a.tensor(false); s.v = a.tensor(false); s.mask = a.tensor(true);
  TORCH_CHECK_TYPE(!a.odd, "query, key, value and attn_mask are tensors");
  s.dropout_p = a.real();
  s.causal = a.flag();
  if (a.i < a.n && a.a[a.i] == Py_None) a.next(); else s.scale = a.real();
  s.gqa = a.flag();
  return s;
}

// sdpa_ops(query, key, value, attn_mask, dropout_p, is_causal, scale, enable_gqa): on the custom ops,
// Philox state from torch's generator; None where the Python route has to take the call
PyObject* py_sdpa_ops(PyObject*, PyObject* const* argv, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  // subclasses (all but Parameter) and function modes may override torch's functions: they have to see the calls of the
  // Python route
  if (at::impl::torch_function_mode_enabled()) Py_RETURN_NONE;
  for (Py_ssize_t i = 0; i < n && i < 4; ++i)
    if (THPVariable_Check(argv[i]) && !THPVariable_CheckTypeExact(Py_TYPE(argv[i]))) Py_RETURN_NONE;
  Args a{argv, n};
  const SdpaArgs in = read_sdpa(a);
  if (traced({&in.q, &in.k, &in.v, &in.mask})) Py_RETURN_NONE;
  Tensor out;
  {
    pybind11::gil_scoped_release no_gil;
    const Sdpa s = prepare(in.q, in.k, in.v, in.mask, in.causal, in.scale, in.gqa, in.dropout_p == 0);
    if (s.key_mask.defined()) {
      out = std::get<0>(key_mask_op().call(s.q, s.k, s.v, s.key_mask, s.scale));
    } else {
      Tensor seed, offset;
      if (in.dropout_p > 0) {
        static const auto op = c10::Dispatcher::singleton().findSchemaOrThrow("aotriton_amd::philox_state", "")
                                   .typed<std::tuple<Tensor, Tensor>(const Tensor&, c10::SymInt)>();
        const int64_t per_row = (s.k.size(2) + 3) / 4;      // Philox counters per query row
        std::tie(seed, offset) = op.call(s.q, s.q.size(0) * s.q.size(1) * s.q.size(2) * per_row);
      } else {
        seed = offset = at::empty({0}, s.q.options().dtype(at::kUInt64));      // not read
      }
      const int64_t edge = in.causal ? (int64_t)FA_WINDOW_TOP_LEFT : 0;
      out = std::get<0>(forward_op().call(s.q, s.k, s.v, s.bias.defined() ? std::optional<Tensor>(s.bias) : std::nullopt,
                                          in.dropout_p, in.causal ? FA_CAUSAL_WINDOWED : FA_CAUSAL_NONE, edge, edge, s.scale,
                                          seed, offset));
    }
  }
  return wrap(out);
  END_HANDLE_TH_ERRORS
}

// sdpa_function(query, key, value, attn_mask, dropout_p, is_causal, scale, enable_gqa, encoded, lse, fillnan, backend,
//               seed, offset1, offset2): on `attention`
PyObject* py_sdpa_function(PyObject*, PyObject* const* argv, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Args a{argv, n};
  const SdpaArgs in = read_sdpa(a);
  AttentionOptions x;
  x.encoded = a.flag();
  x.lse = a.flag();
  x.fillnan = a.flag();
  x.backend = (int)a.integer();
  x.seed = a.word64();
  x.offset1 = a.word64();
  x.offset2 = a.word64();
  Tensor out;
  {
    pybind11::gil_scoped_release no_gil;
    const Sdpa s = prepare(in.q, in.k, in.v, in.mask, in.causal, in.scale, in.gqa);
    x.scale = s.scale;
    x.dropout_p = in.dropout_p;
    if (in.causal) x.mask = Mask{FA_CAUSAL_WINDOWED, FA_WINDOW_TOP_LEFT, FA_WINDOW_TOP_LEFT};
    out = attention(s.q, s.k, s.v, s.bias, x)[0];
  }
  return wrap(out);
  END_HANDLE_TH_ERRORS
}

#define FAST(f) reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(f)), METH_FASTCALL, nullptr
PyMethodDef kMethods[] = {
    {"attn_fwd", FAST(py_attn_fwd)},
    {"attn_bwd", FAST(py_attn_bwd)},
    {"attention", FAST(py_attention)},
    {"attention_varlen", FAST(py_attention_varlen)},
    {"sdpa_ops", FAST(py_sdpa_ops)},
    {"sdpa_function", FAST(py_sdpa_function)},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_torch_host", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__torch_host(void) {
  PyObject* m = PyModule_Create(&kModule);
  if (m != nullptr && PyModule_AddStringConstant(m, "torch_version", FA_TORCH_VERSION) != 0) Py_CLEAR(m);
  return m;
}
