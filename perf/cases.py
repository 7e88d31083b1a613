"""The attention calls a program makes through this library, as cases to be timed.

A case names the entry point it goes through (`api`), the direction (`fwd`, `bwd` or `train` =
forward and backward) and the sizes.  `listed()` has twelve of them, `draw()` makes more of the
same kinds with other sizes.  Tensors are (batch, heads, tokens, head dim) views; `layout` says how
they are stored: `bhsd` contiguous, `bshd` as the transposed view of a (batch, tokens, heads, head dim)
projection or cache.
"""
import math
import random

import numpy as np
import torch

from aotriton_amd import flash, sdpa, torch_ops
from aotriton_amd.autograd import AttentionExtraArgs, attention, attention_varlen

_DTYPES = {'bf16': torch.bfloat16, 'fp16': torch.float16, 'fp32': torch.float32}


def _case(kind, api, do, dtype, B, Hq, Hk, Sq, Sk, D, causal='none', layout='bshd', **more):
    return dict(kind=kind, api=api, do=do, dtype=dtype, B=B, Hq=Hq, Hk=Hk, Sq=Sq, Sk=Sk, D=D, causal=causal,
                layout=layout, **more)


# ---- the kinds of calls ---------------------------------------------------------------------

def _decode(B, Hq, Hk, Sk, D, dtype):
    """One token per sequence against its KV cache (a view of the filled part of the cache)."""
    return _case('decode', 'sdpa_ops', 'fwd', dtype, B, Hq, Hk, 1, Sk, D)


def _chunk(B, Hq, Hk, Sq, Sk, D, dtype):
    """A serving engine's prompt chunk against the cache that already holds what came before it:
    causal, aligned at the bottom right."""
    return _case('chunk', 'operator', 'fwd', dtype, B, Hq, Hk, Sq, Sk, D, causal='bottom_right')


def _prefill(B, Hq, Hk, S, D, dtype, causal='top_left', layout='bhsd'):
    """A whole prompt at once, forward only."""
    return _case('prefill', 'operator', 'fwd', dtype, B, Hq, Hk, S, S, D, causal=causal, layout=layout)


def _encoder(B, H, S, D, dtype):
    """Encoder inference on a padded batch: a boolean key mask through the SDPA entry point."""
    return _case('encoder', 'sdpa_ops', 'fwd', dtype, B, H, H, S, S, D, mask=True)


def _train(B, Hq, Hk, S, D, dtype):
    """Decoder training, forward and backward, through the SDPA entry point and autograd."""
    return _case('train', 'sdpa_ops', 'train', dtype, B, Hq, Hk, S, S, D, causal='top_left')


def _backward(B, Hq, Hk, S, D, dtype, causal='top_left'):
    """The backward operator alone, as a framework's own autograd node calls it."""
    return _case('backward', 'operator', 'bwd', dtype, B, Hq, Hk, S, S, D, causal=causal, layout='bhsd')


def _varlen(n, lo, hi, Hq, Hk, D, dtype, lens_seed):
    """Training on packed sequences of different lengths (n lengths from [lo, hi])."""
    lens = _lengths(n, lo, hi, lens_seed)
    return _case('varlen', 'varlen', 'train', dtype, 1, Hq, Hk, sum(lens), sum(lens), D, causal='top_left',
                 n=n, lo=lo, hi=hi, lens_seed=lens_seed)


def _window(B, H, S, D, dtype, left):
    """Sliding window, additive bias and dropout together, forward and backward operators."""
    return _case('window', 'operator', 'train', dtype, B, H, H, S, S, D, causal='window', layout='bhsd', left=left,
                 bias='given', dropout=0.1)


def _cross(B, H, Sq, Sk, D, dtype):
    """Cross attention with dropout in training: ragged lengths on both sides."""
    return _case('cross', 'sdpa', 'train', dtype, B, H, H, Sq, Sk, D, dropout=0.1)


def _learned_bias(B, H, S, D, dtype):
    """Self attention with an additive bias that is trained: the backward returns its gradient."""
    return _case('learned_bias', 'autograd', 'train', dtype, B, H, H, S, S, D, bias='trained')


def _full_precision(B, H, S, D, causal='none'):
    """fp32 forward and backward."""
    return _case('full_precision', 'autograd', 'train', 'fp32', B, H, H, S, S, D, causal=causal, layout='bhsd')


def listed():
    def named(name, c):
        return dict(c, name=name)
    return [
        # one user's chat at a few thousand tokens: latency of the smallest useful call
        named('decode_one_user', _decode(1, 32, 8, 2051, 128, 'bf16')),
        # a full serving batch at long context: the KV cache is read once, nothing else matters
        named('decode_batch', _decode(32, 32, 8, 8190, 128, 'bf16')),
        # a prompt chunk of a long document
        named('chunked_prefill', _chunk(1, 32, 8, 1024, 16384, 128, 'bf16')),
        # the benchmark's headline forward: B4 H32 S4096 D128 bf16 causal
        named('prefill_4k', _prefill(4, 32, 32, 4096, 128, 'bf16')),
        # sentence encoder on a padded batch
        named('encoder_padded', _encoder(16, 12, 384, 64, 'fp16')),
        # the benchmark's smallest configuration: fp32 (2, 4, 128, 64), forward and backward
        named('fp32_small', _full_precision(2, 4, 128, 64)),
        # a small language model's training step, one layer
        named('train_short', _train(8, 16, 16, 512, 64, 'bf16')),
        # the benchmark's headline backward: B4 H32 S4096 D128 bf16 causal
        named('backward_4k', _backward(4, 32, 32, 4096, 128, 'bf16')),
        # the benchmark's packed configuration: 16 sequences of 256-8192 tokens, Hq 32 / Hkv 8
        named('packed_gqa', _varlen(16, 256, 8192, 32, 8, 128, 'bf16', 1234)),
        # the benchmark's window + bias + dropout configuration: D256 fp16
        named('window_bias_dropout', _window(2, 16, 8192, 256, 'fp16', 1024)),
        # image tokens attending to text and back: odd lengths, a head dim between the usual ones
        named('cross_dropout', _cross(4, 16, 1000, 1531, 80, 'fp16')),
        # relative position bias trained with the model
        named('learned_bias', _learned_bias(8, 12, 512, 64, 'bf16')),
    ]


# ---- more of the same ---------------------------------------------------------------------------

def _log(rng, lo, hi):
    """An integer of [lo, hi], spread over its logarithm; odd ones as often as they come."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


_HEADS = [(32, 8), (32, 32), (16, 16), (64, 8), (24, 8), (40, 40), (12, 12)]


def _drawn(rng):
    kind = rng.choice(['decode', 'decode', 'chunk', 'prefill', 'encoder', 'train', 'train', 'backward', 'varlen',
                       'window', 'cross', 'learned_bias', 'full_precision'])
    half = rng.choice(['bf16', 'bf16', 'fp16'])
    hq, hk = rng.choice(_HEADS)
    if kind == 'decode':
        return _decode(_log(rng, 1, 64), hq, hk, _log(rng, 64, 16384), rng.choice([64, 128, 128, 256]), half)
    if kind == 'chunk':
        sq = _log(rng, 16, 2048)
        return _chunk(_log(rng, 1, 4), hq, hk, sq, sq + _log(rng, 128, 30000), rng.choice([64, 128, 128]), half)
    if kind == 'prefill':
        return _prefill(_log(rng, 1, 8), hq, hk, _log(rng, 128, 16384), rng.choice([64, 96, 128, 128, 256]), half,
                        rng.choice(['top_left', 'top_left', 'none']), rng.choice(['bhsd', 'bshd']))
    if kind == 'encoder':
        return _encoder(_log(rng, 1, 64), rng.choice([8, 12, 16]), _log(rng, 32, 1024), rng.choice([64, 64, 80]), half)
    if kind == 'train':
        return _train(_log(rng, 1, 16), hq, hk, _log(rng, 64, 2048), rng.choice([64, 96, 128]), half)
    if kind == 'backward':
        return _backward(_log(rng, 1, 4), hq, hk, _log(rng, 256, 8192), rng.choice([64, 128, 128, 256]), half,
                         rng.choice(['top_left', 'top_left', 'none']))
    if kind == 'varlen':
        lo = _log(rng, 16, 512)
        return _varlen(_log(rng, 2, 32), lo, _log(rng, 2 * lo, 8192), hq, hk, rng.choice([64, 128, 128]), half,
                       rng.randrange(1 << 30))
    if kind == 'window':
        s = _log(rng, 512, 8192)
        return _window(_log(rng, 1, 2), rng.choice([8, 16]), s, rng.choice([64, 128, 256]), half, max(32, s // rng.choice([2, 4, 8])))
    if kind == 'cross':
        return _cross(_log(rng, 1, 16), rng.choice([8, 16]), _log(rng, 64, 2048), _log(rng, 64, 2048),
                      rng.choice([40, 64, 80, 96, 128]), half)
    if kind == 'learned_bias':
        return _learned_bias(_log(rng, 1, 16), rng.choice([8, 12, 16]), _log(rng, 64, 1024), 64, half)
    return _full_precision(_log(rng, 1, 4), _log(rng, 2, 16), _log(rng, 32, 1024), rng.choice([64, 128]),
                           rng.choice(['none', 'top_left']))


def _cost(case):
    """A yardstick for draw(): seconds at modest rates of this path."""
    w = work(case)
    rate = {'fp32': 2e13, 'bf16': 5e14, 'fp16': 5e14}[case['dtype']] * (0.4 if case.get('dropout') else 1.0)
    return max(w['flops'] / rate, w['bytes'] / 2e12)


def draw(rng):
    """One more case; nothing that costs more than a third of the largest listed one."""
    while True:
        c = _drawn(rng)
        if _cost(c) < 8e-3:
            return c


# ---- inputs -----------------------------------------------------------------------------------

def _lengths(n, lo, hi, seed):
    if seed == 1234:      # the benchmark's own draw
        return [int(x) for x in np.random.default_rng(seed).integers(lo, hi + 1, size=n)]
    r = random.Random(seed)
    return [r.randint(lo, hi) for _ in range(n)]


_CAUSAL = {'none': False, 'top_left': True, 'bottom_right': flash.CausalType.BOTTOM_RIGHT}


def prepare(case, seed):
    dev, dt = torch.device('cuda'), _DTYPES[case['dtype']]
    g = torch.Generator(device=dev).manual_seed(seed)
    B, Hq, Hk, Sq, Sk, D = (case[k] for k in ('B', 'Hq', 'Hk', 'Sq', 'Sk', 'D'))

    def tensor(h, s, room=0):
        if case['layout'] == 'bshd':
            return torch.randn(B, s + room, h, D, device=dev, dtype=dt, generator=g)[:, :s].transpose(1, 2)
        return torch.randn(B, h, s, D, device=dev, dtype=dt, generator=g)

    # a KV cache has room for tokens to come
    room = -Sk % 256 if case['kind'] in ('decode', 'chunk') else 0
    st = dict(case=case, q=tensor(Hq, Sq), k=tensor(Hk, Sk, room), v=tensor(Hk, Sk, room), bias=None,
              scale=1.0 / math.sqrt(D), p=case.get('dropout', 0.0),
              causal=(case['left'], 0) if case['causal'] == 'window' else _CAUSAL[case['causal']])
    if case.get('mask'):
        lens = torch.randint((Sk + 1) // 2, Sk + 1, (B, 1, 1, 1), device=dev, generator=g)
        st['mask'] = torch.arange(Sk, device=dev).view(1, 1, 1, Sk) < lens
    if case.get('bias'):
        st['bias'] = torch.randn(B, Hq, Sq, Sk, device=dev, dtype=dt, generator=g).mul_(0.5)
    if case['do'] != 'fwd':
        st['do'] = tensor(Hq, Sq)
    if case['api'] != 'operator' and case['do'] == 'train':
        st['params'] = [st[k].requires_grad_() for k in ('q', 'k', 'v')]
        if case.get('bias') == 'trained':
            st['params'].append(st['bias'].requires_grad_())
    if case['api'] == 'varlen':
        st['lens'] = np.array(_lengths(case['n'], case['lo'], case['hi'], case['lens_seed']))
    ext = AttentionExtraArgs(philox_seed=0x1234 + seed, philox_offset1=0, philox_offset2=0)
    st['ext'] = ext
    if case['api'] == 'operator':
        u64 = lambda x: torch.tensor([x], device=dev, dtype=torch.int64).view(torch.uint64)
        null = torch.empty([0], device=dev, dtype=torch.uint64)
        st['null'] = null
        st['seed'], st['offset'] = (u64(ext.philox_seed), u64(0)) if st['p'] > 0 else (null, null)
        st['counter'] = torch.zeros([1 if st['causal'] is not False else 0], device=dev, dtype=torch.int32)
        if case['do'] == 'bwd':
            st['o'], st['lse'] = _operator_forward(st)
    return st


# ---- one pass -----------------------------------------------------------------------------------

def _operator_forward(st):
    q, k, v, null = st['q'], st['k'], st['v'], st['null']
    o = torch.empty_like(q)
    lse = torch.empty((q.shape[0] * q.shape[1], q.shape[2]), device=q.device, dtype=torch.float32)
    err = flash.attn_fwd(q, k, v, st['bias'], st['scale'], lse, o, st['p'], st['seed'], st['offset'], 0, null, null,
                         None, st['causal'], st['counter'])
    if err != flash.hipError_t.hipSuccess:
        raise RuntimeError(f'attn_fwd: {err!r}')
    return o, lse


def _operator_backward(st, o, lse):
    q, k, v = st['q'], st['k'], st['v']
    dq, dk, dv = torch.empty_like(q), torch.empty_like(k), torch.empty_like(v)
    err = flash.attn_bwd(q, k, v, st['bias'], st['scale'], o, st['do'], dq, dk, dv, None, flash.lazy_dq_acc(q), lse,
                         flash.lazy_delta(lse), st['p'], st['seed'], st['offset'], 0, st['causal'])
    if err != flash.hipError_t.hipSuccess:
        raise RuntimeError(f'attn_bwd: {err!r}')
    return dq, dk, dv


def run(st):
    case = st['case']
    q, k, v, api, train = st['q'], st['k'], st['v'], case['api'], case['do'] == 'train'
    if api == 'operator':
        if case['do'] == 'bwd':
            return _operator_backward(st, st['o'], st['lse'])
        o, lse = _operator_forward(st)
        return (o, lse) + (_operator_backward(st, o, lse) if train else ())
    with torch.set_grad_enabled(train):
        if api == 'sdpa_ops':
            o = torch_ops.scaled_dot_product_attention(q, k, v, attn_mask=st.get('mask'), is_causal=st['causal'],
                                                       enable_gqa=case['Hq'] != case['Hk'])
        elif api == 'sdpa':
            o = sdpa.scaled_dot_product_attention(q, k, v, dropout_p=st['p'], is_causal=st['causal'], extra=st['ext'])
        elif api == 'autograd':
            o = attention(q, k, v, st['bias'], st['causal'], st['scale'], st['p'], st['ext'])[0]
        else:
            o = attention_varlen(q, k, v, st['lens'], st['lens'], st['causal'], st['scale'], st['p'], st['ext'])[0]
    if not train:
        return o
    return (o,) + torch.autograd.grad(o, st['params'], st['do'])


# ---- what a pass cannot do without ----------------------------------------------------------------

def _pairs(case):
    """Visible (query, key) pairs of one head of one batch element (all sequences of a packed one)."""
    def triangle(sq, sk, shift):
        # row i sees keys 0 .. min(i + shift, sk - 1)
        rows = max(0, min(sq, sk - shift))
        return rows * (1 + shift) + rows * (rows - 1) // 2 + (sq - rows) * sk
    sq, sk = case['Sq'], case['Sk']
    if case['kind'] == 'varlen':
        return sum(triangle(n, n, 0) for n in _lengths(case['n'], case['lo'], case['hi'], case['lens_seed']))
    if case['causal'] == 'top_left':
        return triangle(sq, sk, 0)
    if case['causal'] == 'bottom_right':
        return triangle(sq, sk, sk - sq)
    if case['causal'] == 'window':
        w = min(case['left'], sk)
        return triangle(sq, sk, 0) - triangle(max(0, sq - w - 1), sk, 0)
    return sq * sk


def work(case):
    B, Hq, Hk, Sq, Sk, D = (case[k] for k in ('B', 'Hq', 'Hk', 'Sq', 'Sk', 'D'))
    size = 4 if case['dtype'] == 'fp32' else 2
    pairs = _pairs(case) * B * Hq
    q, kv, stats = B * Hq * Sq * D * size, 2 * B * Hk * Sk * D * size, B * Hq * Sq * 4
    bias = pairs * size if case.get('bias') else B * Sk if case.get('mask') else 0
    forward, n_bytes = 4.0 * pairs * D, q + kv + bias
    if case['do'] == 'fwd':
        return dict(bytes=n_bytes + q + stats, flops=forward)
    n_bytes += q + q + kv + (bias if case.get('bias') == 'trained' else 0)      # dO; dQ, dK and dV, dB
    if case['do'] == 'bwd':
        return dict(bytes=n_bytes + q + stats, flops=2.5 * forward)          # reads O and its statistics
    return dict(bytes=n_bytes + q, flops=3.5 * forward)                         # writes O


def tolerance(case):
    # sums are fp32 throughout; P and dS are rounded to the tensors' type once, and so are the results
    return {'fp32': {'rel': 1e-5, 'max': 1e-3}, 'fp16': {'rel': 2e-3, 'max': 0.08}, 'bf16': {'rel': 1e-2, 'max': 0.4}}[case['dtype']]
