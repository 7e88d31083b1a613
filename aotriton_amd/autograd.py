"""torch.autograd Functions over the flash operators.

Counterpart of modules/flash/tests/attn_torch_function.py:87-270 and
varlen_attn_torch_function.py:38-206: same allocation shapes (O (B,Hq,Sq,Dv); LSE
(B*Hq, Sq) dense, (Hq, total_q) compact), the reference's default philox seed and offsets,
and the backward reading the forward's *output* seed/offset with offset2 = 0.  The Functions
themselves are native (csrc/torch/host.cpp).
"""
from dataclasses import dataclass

import numpy as np

from . import _host
from .flash import translate_causal

_torch_host = _host.load()

DEFAULT_PHILOX_SEED = 0x1BF52
DEFAULT_PHILOX_OFFSET_1 = 0x1D4000
DEFAULT_PHILOX_OFFSET_2 = 0x000B42


@dataclass
class AttentionExtraArgs:
    return_encoded_softmax: bool = False
    return_logsumexp: bool = False
    fillnan: bool = False
    bwd_backend: int = -1          # -1 library's choice, 0 split, 1 fused
    philox_seed: int = DEFAULT_PHILOX_SEED
    philox_offset1: int = DEFAULT_PHILOX_OFFSET_1
    philox_offset2: int = DEFAULT_PHILOX_OFFSET_2


_DEFAULTS = AttentionExtraArgs()


def _extra_args(ext):
    """What the native functions take of an AttentionExtraArgs, in their order."""
    return (ext.return_encoded_softmax, ext.return_logsumexp, ext.fillnan, ext.bwd_backend, ext.philox_seed,
            ext.philox_offset1, ext.philox_offset2)


def attention(q, k, v, b, causal, sm_scale, dropout_p, ext=None):
    """(Out, encoded softmax or None, logsumexp or None), differentiable in q, k, v and b."""
    return _torch_host.attention(q, k, v, b, *translate_causal(causal), sm_scale, dropout_p, *_extra_args(ext or _DEFAULTS))


def _lengths(seqlens):
    """A host array of any shape and number type as the list of ints that the native function reads."""
    return np.asarray(seqlens).reshape(-1).astype(np.int64).tolist()


def attention_varlen(q, k, v, seqlens_q, seqlens_k, causal, sm_scale, dropout_p, ext=None):
    """Compact varlen: q (1, Hq, total_q, D), k/v (1, Hk, total_k, D); the lengths are host arrays that add
    up to total_q and total_k (ValueError otherwise)."""
    return _torch_host.attention_varlen(q, k, v, _lengths(seqlens_q), _lengths(seqlens_k),
                                        *translate_causal(causal), sm_scale, dropout_p, *_extra_args(ext or _DEFAULTS))
