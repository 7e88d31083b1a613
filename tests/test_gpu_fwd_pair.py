"""Forward at head dims above 128 by pairs of waves (fa_fwd_pair.h), against the oracle where its steps and stages can go wrong: fewer units
than stages, row blocks without rows or without visible keys, masked units at both ends, moved references, bias rows anywhere."""
import math

import pytest
import torch

from test_gpu_attention import _run_case
from test_launch_queries import fwd
from oracle import fa_ref
from _util import FUDGE, check, make_inputs

BF, HF = torch.bfloat16, torch.float16


def test_short_calls_of_several_row_blocks():
    """tiles where one round of them is shorter than the packed rows' steps; one row block stays packed"""
    for call in [(1, 8, 2, 512, 512, 256, True), (8, 16, 16, 64, 300, 256), (1, 8, 2, 256, 256, 256, True), (4, 16, 16, 60, 60, 200)]:
        assert not fwd(*call).flags & 128, call
    for call in [(1, 16, 4, 256, 1024, 256), (1, 32, 32, 128, 2000, 256), (1, 32, 8, 1, 64, 256), (4, 16, 16, 16, 100, 256), (4, 16, 16, 32, 60, 256)]:
        assert fwd(*call).flags & 128, call


CASES = [
    # B, Hq, Hk, Sq, Sk, D, Dv, dtype, causal, dropout, bias
    (2, 2, 2, 17, 1, 256, 256, BF, False, 0.0, False),             # one key, three row blocks without rows
    (2, 4, 2, 33, 32, 256, 256, HF, False, 0.3, True),             # one whole unit
    (1, 4, 4, 128, 33, 256, 256, BF, False, 0.1, False),           # two units
    (2, 2, 1, 129, 96, 256, 256, HF, False, 0.0, True),            # as many units as stages
    (2, 2, 1, 160, 97, 256, 256, BF, False, 0.2, True),
    (1, 4, 2, 300, 300, 256, 256, HF, True, 0.0, False),
    (1, 4, 2, 257, 390, 256, 256, BF, True, 0.25, True),
    (1, 2, 2, 390, 257, 256, 256, HF, (-140, 200), 0.0, True),     # rows that see nothing
    (1, 2, 1, 515, 520, 256, 256, BF, (60, 90), 0.3, True),        # masked units on both sides, skipped ones on the left
    (1, 2, 1, 515, 520, 256, 256, HF, (40, -8), 0.0, False),
    (2, 4, 2, 260, 392, 136, 136, BF, True, 0.1, True),            # head dims rounded up
    (1, 4, 2, 129, 200, 200, 248, HF, False, 0.0, False),
    (1, 2, 2, 270, 264, 248, 160, BF, (40, 20), 0.2, True),
]


@pytest.mark.gpu
@pytest.mark.parametrize('case', CASES, ids=lambda c: '-'.join(str(x).replace('torch.', '') for x in c))
def test_pairs_meet_the_oracle(case):
    B, Hq, Hk, Sq, Sk, D, Dv, dtype, causal, p, bias = case
    x = fwd(B, Hq, Hk, Sq, Sk, max(D, Dv), causal, p, bias)
    assert (x.block_m, x.block_n, x.num_waves) == (128, 32, 8)
    _run_case(B, Hq, Hk, Sq, Sk, D, dtype, causal, dropout_p=p, bias=bias, seed=23, Dv=Dv)


def _forward(q, k, v, b, causal, sm):
    from aotriton_amd import flash
    o = torch.full((*q.shape[:-1], v.shape[-1]), float('nan'), device='cuda', dtype=q.dtype)
    lse = torch.full((q.shape[0] * q.shape[1], q.shape[2]), float('nan'), device='cuda')
    null = torch.empty(0, device='cuda', dtype=torch.int64)
    err = flash.attn_fwd(q, k, v, b, sm, lse, o, 0.0, null, null, 0, null, null, None, causal, torch.zeros(1, device='cuda', dtype=torch.int32))
    assert err == flash.hipError_t.hipSuccess
    torch.cuda.synchronize()
    return o, lse.view(q.shape[0], q.shape[1], -1)


@pytest.mark.gpu
@pytest.mark.parametrize('dtype,causal,sm,bias', [(BF, False, 1 / 16, False), (HF, True, 1 / 16, True), (BF, False, -1 / 16, False), (HF, False, 1.0, False)])
def test_references_that_move(dtype, causal, sm, bias):
    """Scores that grow along the keys (every few units the exponentials leave their range and a unit is done in full), for some rows
    only; a negative scale; scores past the range in which the scale is folded into the exponent."""
    q, k, v, b, _ = make_inputs(1, 2, 2, 200, 700, 256, dtype, 'cuda', seed=5, bias=bias)
    k *= (torch.arange(700, device='cuda') / 100)[None, None, :, None].to(dtype)
    q[:, :, ::3] *= 0.05
    o, lse = _forward(q, k, v, b if bias else torch.empty(0, 0, 0, 0, device='cuda', dtype=dtype), causal, sm)
    from aotriton_amd import flash
    ct, wl, wr = flash.translate_causal(causal)
    f = lambda t: t.float()
    ro, rl, _ = fa_ref.attn_fwd_ref(f(q), f(k), f(v), f(b) if bias else None, sm, ct, wl, wr, 0.0, None)
    lo, _, _ = fa_ref.attn_fwd_ref(q, k, v, b if bias else None, sm, ct, wl, wr, 0.0, None)
    check('out', o, ro, lo, FUDGE['out'])
    # fp32 sums of 256 products, each term rounded to 2^-24 of it
    assert ((lse - rl.view_as(lse)).abs() <= 1e-5 * (1 + rl.view_as(lse).abs()) + 2e-4).all()


@pytest.mark.gpu
@pytest.mark.parametrize('kind', ['offset', 'odd rows', 'broadcast rows'])
def test_bias_layouts_agree(kind):
    """A bias gives the same bits wherever its rows lie."""
    B, H, Sq, Sk = 1, 2, 190, 230
    q, k, v, b, _ = make_inputs(B, H, H, Sq, Sk, 256, BF, 'cuda', seed=6, bias=True)
    if kind == 'broadcast rows':
        b = b[:, :, :1].expand(B, H, Sq, Sk)
    want, wl = _forward(q, k, v, b.contiguous(), (100, 30), 1 / 16)
    if kind == 'offset':
        x = torch.empty(B * H * Sq * Sk + 1, device='cuda', dtype=BF)[1:].view(B, H, Sq, Sk).copy_(b)
    elif kind == 'odd rows':
        x = torch.empty(B, H, Sq, Sk + 3, device='cuda', dtype=BF)[..., :Sk].copy_(b)
    else:
        x = b
    got, gl = _forward(q, k, v, x, (100, 30), 1 / 16)
    assert torch.equal(got, want) and torch.equal(gl, wl)


@pytest.mark.gpu
@pytest.mark.parametrize('p,causal', [(0.0, False), (0.25, (100, 30))])
def test_columns_of_a_bias_apart(p, causal):
    """Columns that lie apart, which the views of the bindings take, go through the units' general step: adjacent columns' results but
    for the roundings of P."""
    from aotriton_amd import flash
    from aotriton_amd.pyaotriton import T4
    B, H, Sq, Sk = 1, 3, 190, 261
    q, k, v, b, _ = make_inputs(B, H, H, Sq, Sk, 256, BF, 'cuda', seed=6, bias=True)
    b = b.contiguous()
    seed, off = (torch.tensor([x], device='cuda', dtype=torch.uint64) for x in (7, 8))
    null, out = torch.empty([0], device='cuda', dtype=torch.uint64), []
    for x in (b, b.transpose(2, 3).contiguous().transpose(2, 3)):
        o, L = torch.empty_like(q), torch.empty(B * H, Sq, device='cuda')
        params = flash.fa_forward_op_params()
        flash._fill_fwd(params, q, k, v, None, 1 / 16, L, o, p, seed, off, 0, null, null, None, causal, null)
        params.B = T4(x.data_ptr(), tuple(x.size()), x.stride(), flash.cast_dtype(BF))
        params.varlen_type = 0
        assert flash.fa_forward_op(params, params.kVersion, flash._stream(), None) == flash.hipError_t.hipSuccess
        torch.cuda.synchronize()
        out.append((o.float(), L))
    (o, L), (o1, L1) = out
    # P rounded to 16 bits on either side (2^-9 of values that sum to 1 / (1 - p)), the results too
    assert ((o - o1).abs() <= 2 ** -8 * (1 / (1 - p) * v.float().abs().max() + o.abs())).all()
    seen = torch.isfinite(L)
    assert torch.equal(seen, torch.isfinite(L1)) and (L - L1).abs()[seen].max() <= 1e-5


@pytest.mark.gpu
@pytest.mark.parametrize('causal', [False, True])
def test_packed_sequences(causal):
    """Lengths around tiles and units, walked by level, against 64 bits."""
    from aotriton_amd.autograd import attention_varlen, AttentionExtraArgs
    lens, H = [1, 31, 32, 33, 127, 128, 129, 260, 640, 65], 8
    g = torch.Generator(device='cuda').manual_seed(9)
    q, k, v = (torch.randn(1, H, sum(lens), 256, device='cuda', generator=g).to(BF) for _ in range(3))
    got = attention_varlen(q, k, v, lens, lens, causal, 1 / 16, 0.0, AttentionExtraArgs(return_logsumexp=False))[0]
    at = 0
    for n in lens:
        x, y, z = (t[:, :, at:at + n].double() for t in (q, k, v))
        s = torch.matmul(x, y.transpose(-1, -2).contiguous()) / 16
        if causal:
            s = s.masked_fill(torch.ones(n, n, device='cuda', dtype=torch.bool).triu(1), float('-inf'))
        want = torch.matmul(torch.softmax(s, -1), z)
        # P rounded to 16 bits, the result rounded
        assert ((got[:, :, at:at + n].double() - want).norm() / want.norm()).item() < 3 * torch.finfo(BF).eps / 2, n
        at += n
