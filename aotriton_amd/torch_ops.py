"""torch.library registration of the flash operators.

`torch.ops.aotriton_amd.flash_attention_forward / flash_attention_backward` are custom ops
(kernels and autograd formula in csrc/torch/host.cpp) with fake (shape-only) implementations,
so that code using them can be traced by torch.compile / AOTAutograd.

    flash_attention_forward(q, k, v, bias, dropout_p, causal_type, window_left, window_right, sm_scale, seed, offset)
        -> Out (B, Hq, Sq, Dv), logsumexp (B*Hq, Sq) fp32
    flash_attention_forward_key_mask(q, k, v, mask, sm_scale)
        -> the same, under a boolean (B or 1, Hq or 1, 1, Sk) mask that the kernels read as it is
    flash_attention_backward(dout, q, k, v, bias, out, lse, dropout_p, causal_type, window_left, window_right,
                             sm_scale, seed, offset, need_dbias, backend)
        -> dQ, dK, dV, dB (empty unless need_dbias); backend: -1 the library's choice, 0 split, 1 fused
    philox_state(like, increment)
        -> seed and offset (uint64[1] tensors on like's device) of the device's default generator, whose
           offset moves on by `increment` counters (rounded up to a multiple of 4)

They take what PyTorch's ROCm SDPA puts
into attn_fwd_params / attn_bwd_params (include/aotriton/flash.h:96-174 of the
reference): (B, H, S, D) tensors with unit last stride, an optional additive bias,
causal type with window sentinels, and the Philox seed / offset as uint64[1] device
tensors.  `philox_state` works the way the ROCm SDPA takes them from the generator's philox state.
It reads and advances host-side generator state, so it is tagged as a seeded random op: graph
passes must not merge two calls or recompute one.  Under HIP graph capture the host read happens
once, at capture: every replay would reuse the captured seed and offset.  Callers that replay
graphs pass their own seed / offset tensors to flash_attention_forward and update them on the
device between replays.

`scaled_dot_product_attention` here has the signature of
torch.nn.functional.scaled_dot_product_attention and runs on those ops.
"""
import torch
from torch import Tensor

from . import _host
from .flash import WindowValue
from .sdpa import prepare

_torch_host = _host.load()      # registers the ops

__all__ = ['flash_attention_forward', 'flash_attention_backward', 'philox_state', 'scaled_dot_product_attention']


philox_state = torch.ops.aotriton_amd.philox_state
flash_attention_forward = torch.ops.aotriton_amd.flash_attention_forward
flash_attention_backward = torch.ops.aotriton_amd.flash_attention_backward


@torch.library.register_fake('aotriton_amd::philox_state')
def _(like, increment):
    return (torch.empty([1], device=like.device, dtype=torch.uint64),
            torch.empty([1], device=like.device, dtype=torch.uint64))


@torch.library.register_fake('aotriton_amd::flash_attention_forward')
def _(q, k, v, bias, dropout_p, causal_type, window_left, window_right, sm_scale, philox_seed, philox_offset):
    o = torch.empty((q.shape[0], q.shape[1], q.shape[2], v.shape[3]), device=q.device, dtype=q.dtype)
    lse = torch.empty((q.shape[0] * q.shape[1], q.shape[2]), device=q.device, dtype=torch.float32)
    return o, lse


@torch.library.register_fake('aotriton_amd::flash_attention_forward_key_mask')
def _(q, k, v, mask, sm_scale):
    o = torch.empty((q.shape[0], q.shape[1], q.shape[2], v.shape[3]), device=q.device, dtype=q.dtype)
    lse = torch.empty((q.shape[0] * q.shape[1], q.shape[2]), device=q.device, dtype=torch.float32)
    return o, lse


@torch.library.register_fake('aotriton_amd::flash_attention_backward')
def _(dout, q, k, v, bias, out, lse, dropout_p, causal_type, window_left, window_right, sm_scale, philox_seed,
      philox_offset, need_dbias, backend):
    mk = lambda t: torch.empty(t.shape, device=q.device, dtype=q.dtype)
    want_db = need_dbias and bias is not None
    return mk(q), mk(k), mk(v), (mk(bias) if want_db else torch.empty([0], device=q.device, dtype=q.dtype))


def scaled_dot_product_attention(query, key, value, attn_mask=None, dropout_p=0.0, is_causal=False,
                                 scale=None, enable_gqa=False):
    """torch.nn.functional.scaled_dot_product_attention on the custom ops above: 4-D fp16/bf16
    CUDA tensors (B, H, L, E), head dims up to 512 (multiples of 8 for the MFMA kernels).  A boolean mask becomes an
    additive one (0 / -inf); a query row that the mask hides completely yields zeros instead
    of NaN; dropout draws seed and offset from torch's CUDA generator (so torch.manual_seed
    governs it) but uses the operators' Philox stream, not the one of torch's own kernels.
    As in torch, is_causal means the top-left aligned lower triangle.
    """
    if not torch.compiler.is_compiling():
        out = _torch_host.sdpa_ops(query, key, value, attn_mask, dropout_p, is_causal, scale, enable_gqa)
        if out is not None:      # None: subclasses, function and dispatch modes, functorch transforms
            return out
    q, k, v, bias, sm_scale = prepare(query, key, value, attn_mask, is_causal, scale, enable_gqa)
    hq = q.shape[1]
    if dropout_p > 0.0:
        stride = (k.shape[2] + 3) // 4          # Philox counters per query row
        seed, offset = torch.ops.aotriton_amd.philox_state(q, q.shape[0] * hq * q.shape[2] * stride)
    else:
        seed = offset = torch.zeros([1], device=q.device, dtype=torch.int64).view(torch.uint64)
    ct = 3 if is_causal else 0
    wl = wr = int(WindowValue.TOP_LEFT_ALIGNED) if is_causal else 0
    o, _ = torch.ops.aotriton_amd.flash_attention_forward(q, k, v, bias, float(dropout_p), ct, wl, wr, sm_scale,
                                                          seed, offset)
    return o


# ---- routing torch.nn.functional.scaled_dot_product_attention itself --------------------------
# The consumer the reference names is PyTorch's SDPA on ROCm (README.md:71-75 of the reference):
# callers write F.scaled_dot_product_attention and the dispatcher picks the flash backend.  The
# two hooks below give the same effect without touching callers: `sdpa_router()` is a
# TorchFunctionMode (scoped, composes with torch.compile's tracing of the custom ops), `install()`
# replaces the attribute on torch.nn.functional for code that cannot be wrapped in a `with`.
def _routable(query, key, value, attn_mask, dropout_p, enable_gqa=False):
    ts = (query, key, value)
    if not all(isinstance(t, Tensor) and t.is_cuda and t.dim() == 4 for t in ts):
        return False
    if query.dtype not in (torch.float16, torch.bfloat16, torch.float32):
        return False
    if not (key.dtype == query.dtype and value.dtype == query.dtype):
        return False
    dqk, dv = query.shape[-1], value.shape[-1]
    # (head dims that are no multiple of 8 would run on the element-wise kernels: correct but slow, so the
    # router leaves them to torch; scaled_dot_product_attention above takes them when called directly)
    if dqk % 8 or dv % 8 or dqk > 512 or dv > 512 or key.shape[-1] != dqk:
        return False
    if query.shape[1] % max(key.shape[1], 1) or key.shape[1] != value.shape[1]:
        return False
    # unequal head counts are grouped-query attention only when the caller says so (torch raises otherwise)
    if query.shape[1] != key.shape[1] and not enable_gqa:
        return False
    # what the operators would reject goes to torch, which raises its own error or broadcasts
    if not (query.shape[0] == key.shape[0] == value.shape[0]) or key.shape[2] != value.shape[2]:
        return False
    if not (query.device == key.device == value.device):
        return False
    if attn_mask is not None and (not isinstance(attn_mask, Tensor) or attn_mask.device != query.device):
        return False
    if getattr(query, 'is_nested', False) or getattr(key, 'is_nested', False):
        return False
    return True


_torch_sdpa = torch.nn.functional.scaled_dot_product_attention


def _dispatch(query, key, value, attn_mask=None, dropout_p=0.0, is_causal=False, scale=None, enable_gqa=False):
    if _routable(query, key, value, attn_mask, dropout_p, enable_gqa):
        return scaled_dot_product_attention(query, key, value, attn_mask, dropout_p, is_causal, scale, enable_gqa)
    return _torch_sdpa(query, key, value, attn_mask=attn_mask, dropout_p=dropout_p, is_causal=is_causal,
                       scale=scale, enable_gqa=enable_gqa)


class sdpa_router(torch.overrides.TorchFunctionMode):
    """`with sdpa_router(): ...` sends every F.scaled_dot_product_attention call on 4-D CUDA
    fp16/bf16/fp32 tensors (head dims multiples of 8 up to 512) to this library's operators;
    anything else falls through to PyTorch's own implementation."""

    def __torch_function__(self, func, types, args=(), kwargs=None):
        kwargs = kwargs or {}
        if func is _torch_sdpa:
            with torch._C.DisableTorchFunction():
                return _dispatch(*args, **kwargs)
        return func(*args, **kwargs)


def install():
    """Make torch.nn.functional.scaled_dot_product_attention route here process-wide
    (undo with uninstall()).  Modules that bound the function at import time keep the original;
    for those use the sdpa_router() mode."""
    torch.nn.functional.scaled_dot_product_attention = _dispatch


def uninstall():
    torch.nn.functional.scaled_dot_product_attention = _torch_sdpa
