"""dK/dV with a bias whose rows are whole aligned 16-byte pieces take a kernel of their own: to the bit the results of the
kernel for any layout, given the same bias with an odd row stride; and dropout whose scale lies in the row statistics,
against the oracle at probabilities near both ends."""
import math

import pytest
import torch

from test_gpu_attention import _run_case
from test_launch_queries import bwd
from _util import make_inputs

pytestmark = pytest.mark.gpu

BF, HF = torch.bfloat16, torch.float16


@pytest.mark.parametrize('D', [64, 80, 128, 256])
@pytest.mark.parametrize('Sq,Sk,causal,p', [(70, 72, False, 0.0), (300, 136, True, 0.1), (257, 520, (60, 90), 0.3), (129, 264, (40, -5), 0.0)])
def test_aligned_rows_give_the_bits_of_the_general_kernel(D, Sq, Sk, causal, p):
    from aotriton_amd import flash
    Hq, Hk, dt = 6, 2, HF
    B = 2 ** 23 // (Hq * Sq * Sk) + 1      # large enough for the stored dS
    q, k, v, _, do = make_inputs(B, Hq, Hk, Sq, Sk, D, dt, 'cuda', seed=9)
    b = torch.randn(B, Hq, Sq, Sk, device='cuda', dtype=dt)
    odd = torch.empty(B, Hq, Sq, Sk + 3, device='cuda', dtype=dt)[..., 1:Sk + 1].copy_(b)
    seed = torch.tensor([77], device='cuda', dtype=torch.uint64)
    off = torch.tensor([5], device='cuda', dtype=torch.uint64)
    null = torch.empty([0], device='cuda', dtype=torch.uint64)
    rng = (seed, off) if p else (null, null)
    sm, out = 1 / math.sqrt(D), []
    o, L = torch.empty_like(q), torch.empty(B * Hq, Sq, device='cuda')
    assert flash.attn_fwd(q, k, v, b, sm, L, o, p, *rng, 0, null, null, None, causal, null) == flash.hipError_t.hipSuccess
    for bias in (b, odd):
        dq, dk, dv = torch.empty_like(q), torch.empty_like(k), torch.empty_like(v)
        err = flash.attn_bwd(q, k, v, bias, sm, o, do, dq, dk, dv, None, flash.lazy_dq_acc(q), L, flash.lazy_delta(L), p, *rng,
                             0, causal)
        assert err == flash.hipError_t.hipSuccess
        out.append((dq, dk, dv))
    for x, y in zip(*out):
        assert torch.isfinite(x).all() and torch.equal(x, y)


@pytest.mark.parametrize('p', [0.003, 0.5, 0.97])
@pytest.mark.parametrize('D,bias', [(64, True), (80, False), (128, True), (256, False)])
def test_dropout_scale_in_the_row_statistics(D, bias, p):
    _run_case(4, 6, 3, 260, 200, D, BF, True, dropout_p=p, bias=bias, seed=31)


@pytest.mark.parametrize('D,dt', [(64, BF), (128, HF), (256, HF)])
@pytest.mark.parametrize('Sq,Sk,causal,p', [(40, 7, False, 0.0), (70, 9, False, 0.1), (200, 131, True, 0.0), (129, 257, (60, 90), 0.2)])
@pytest.mark.parametrize('keep', [True, False])
def test_rows_at_any_alignment(D, dt, Sq, Sk, causal, p, keep):
    """rows that start anywhere and end inside a piece, against the oracle, with and without a workspace"""
    from aotriton_amd._lib import lib
    lib.fa_set_bwd_workspace_limit(-1 if keep else 0)
    try:
        _run_case(3, 4, 2, Sq, Sk, D, dt, causal, dropout_p=p, bias=True, bias_layout='odd', seed=12)
    finally:
        lib.fa_set_bwd_workspace_limit(-1)


@pytest.mark.parametrize('D', [64, 128, 256])
@pytest.mark.parametrize('Sq,Sk,causal,p', [(70, 299, False, 0.0), (161, 128, True, 0.1), (33, 257, (20, 100), 0.0)])
def test_db_rows_at_any_alignment(D, Sq, Sk, causal, p):
    """odd bias and dB rows against rows that start at 16-byte boundaries: the same bits, nothing written beside them"""
    from aotriton_amd import flash
    from aotriton_amd._lib import lib
    B, H, dt = 2, 3, BF
    q, k, v, _, do = make_inputs(B, H, H, Sq, Sk, D, dt, 'cuda', seed=14)
    seed, off = (torch.tensor([x], device='cuda', dtype=torch.uint64) for x in (7, 8))
    null, sm, out = torch.empty([0], device='cuda', dtype=torch.uint64), 1 / math.sqrt(D), []
    values = torch.randn(B, H, Sq, Sk, device='cuda', dtype=dt)
    lib.fa_set_bwd_workspace_limit(0)
    try:
        for width in ((Sk + 7) // 8 * 8, Sk + (1 - Sk % 2) + 2):
            b, db = (torch.full((B * H * Sq * width + 8,), x, device='cuda', dtype=dt) for x in (float('nan'), 7.0))
            at = 0 if width % 8 == 0 else 1
            view = lambda t: t[at:at + B * H * Sq * width].view(B, H, Sq, width)[..., :Sk]
            view(b).copy_(values)
            o, L = torch.empty_like(q), torch.empty(B * H, Sq, device='cuda')
            assert flash.attn_fwd(q, k, v, values, sm, L, o, p, seed, off, 0, null, null, None, causal, null) == flash.hipError_t.hipSuccess
            dq, dk, dv = torch.empty_like(q), torch.empty_like(k), torch.empty_like(v)
            err = flash.attn_bwd(q, k, v, view(b), sm, o, do, dq, dk, dv, view(db), flash.lazy_dq_acc(q), L, flash.lazy_delta(L), p,
                                 seed, off, 0, causal)
            assert err == flash.hipError_t.hipSuccess
            got = view(db).clone()
            view(db).fill_(7.0)
            assert (db == 7.0).all()
            out.append((dq, dk, dv, got))
    finally:
        lib.fa_set_bwd_workspace_limit(-1)
    for x, y in zip(*out):
        assert torch.isfinite(x).all() and torch.equal(x, y)


@pytest.mark.parametrize('D', [136, 200, 248])
@pytest.mark.parametrize('dt', [BF, HF])
@pytest.mark.parametrize('Sq,Sk,causal,p', [(40, 136, (60, 90), 0.0), (300, 136, True, 0.0), (70, 72, (40, -5), 0.0), (129, 264, False, 0.0),
                                            (129, 264, True, 0.2)])
@pytest.mark.parametrize('layout', ['padded', 'odd'])
def test_recomputed_dq_at_padded_head_dims(D, dt, Sq, Sk, causal, p, layout):
    """dQ and dB without a workspace, head dims rounded up to 256 columns: every lane stores through its own pointer"""
    from aotriton_amd._lib import lib
    lib.fa_set_bwd_workspace_limit(0)
    try:
        _run_case(2, 4, 2, Sq, Sk, D, dt, causal, dropout_p=p, bias=True, bias_layout=layout, seed=23)
    finally:
        lib.fa_set_bwd_workspace_limit(-1)


@pytest.mark.parametrize('D', [40, 64, 128, 256])
@pytest.mark.parametrize('Sq,Sk,causal,p', [(70, 136, False, 0.0), (300, 131, True, 0.0), (257, 520, (60, 90), 0.0), (129, 261, False, 0.1),
                                            (65, 9, False, 0.0)])
def test_stored_ds_under_rows_at_any_alignment(D, Sq, Sk, causal, p):
    """The backward that keeps dS and writes dB from it, given the same bias and the same dB in rows that start at 16-byte
    boundaries and in odd ones: the same bits, nothing written beside dB's rows."""
    from aotriton_amd import flash
    H, dt = 6, BF
    B = 2 ** 22 // (H * Sq * Sk) + 1      # large enough for the stored dS
    q, k, v, _, do = make_inputs(B, H, H, Sq, Sk, D, dt, 'cuda', seed=15)
    seed, off = (torch.tensor([x], device='cuda', dtype=torch.uint64) for x in (7, 8))
    null, sm, out = torch.empty([0], device='cuda', dtype=torch.uint64), 1 / math.sqrt(D), []
    values = torch.randn(B, H, Sq, Sk, device='cuda', dtype=dt)
    o, L = torch.empty_like(q), torch.empty(B * H, Sq, device='cuda')
    assert flash.attn_fwd(q, k, v, values, sm, L, o, p, seed, off, 0, null, null, None, causal, null) == flash.hipError_t.hipSuccess
    odd = Sk + (1 - Sk % 2) + 2
    for width, at in (((Sk + 7) // 8 * 8, 0), (odd, 1)):
        b = torch.full((B * H * Sq * width + 8,), float('nan'), device='cuda', dtype=dt)
        view = lambda t: t[at:at + B * H * Sq * width].view(B, H, Sq, width)[..., :Sk]
        view(b).copy_(values)
        db = torch.full_like(b, 7.0)
        dq, dk, dv = torch.empty_like(q), torch.empty_like(k), torch.empty_like(v)
        strides = view(db).stride()
        assert bwd(1, B, H, H, Sq, Sk, D, causal, p, bias=strides, db=True, at=2 * at).flags & 16
        err = flash.attn_bwd(q, k, v, view(b), sm, o, do, dq, dk, dv, view(db), flash.lazy_dq_acc(q), L,
                             flash.lazy_delta(L), p, seed, off, 0, causal)
        assert err == flash.hipError_t.hipSuccess
        out.append((dq, dk, dv, view(db).clone()))
        view(db).fill_(7.0)
        assert (db == 7.0).all()
    for x, y in zip(*out):
        assert torch.isfinite(x).all() and torch.equal(x, y)


@pytest.mark.parametrize('B,H,Sq,Sk,causal,layout', [(1, 8, 1024, 1024, False, 'padded'), (1, 5, 1000, 1023, True, 'odd'),
                                                     (1, 5, 1024, 1000, (600, 400), 'odd')])
def test_parts_with_a_bias(B, H, Sq, Sk, causal, layout):
    """dK/dV items that store dS cut into parts, several to a CU, at D = 64 with a bias: against the oracle"""
    assert bwd(1, B, H, H, Sq, Sk, 64, causal, bias=True, db=True).flags & 80 == 80
    _run_case(B, H, H, Sq, Sk, 64, BF, causal, bias=True, bias_layout=layout, seed=33)


@pytest.mark.parametrize('stored', [True, False])
@pytest.mark.parametrize('D,dt,B,H,Sq,Sk,causal', [(256, HF, 1, 4, 520, 261, False), (256, BF, 1, 4, 300, 261, True),
                                                   (256, HF, 1, 3, 300, 9, False), (200, BF, 2, 3, 520, 136, True),
                                                   (200, HF, 1, 4, 300, 389, (100, 30)), (256, BF, 1, 2, 260, 7, False)])
@pytest.mark.parametrize('layout', ['padded', 'odd'])
def test_rows_of_a_bias_with_dropout(D, dt, B, H, Sq, Sk, causal, layout, stored):
    """256 columns, bias and dropout: dK/dV items cut into parts, and items that recompute dS without a workspace, whose bias has
    rows of unit stride (fewer than eight keys: one of any layout)"""
    from aotriton_amd._lib import lib
    lib.fa_set_bwd_workspace_limit(-1 if stored else 0)
    try:
        assert bwd(1, B, H, H, Sq, Sk, D, causal, 0.2, bias=True).flags & 80 == (80 if stored else 0)
        _run_case(B, H, H, Sq, Sk, D, dt, causal, dropout_p=0.2, bias=True, bias_layout=layout, seed=35)
    finally:
        lib.fa_set_bwd_workspace_limit(-1)


@pytest.mark.parametrize('D', [200, 256])
@pytest.mark.parametrize('stored', [True, False])
def test_columns_of_a_bias_apart_with_dropout(D, stored):
    """the same with the columns of the bias apart, which the views of the bindings take: the bits of adjacent columns"""
    from aotriton_amd import flash
    from aotriton_amd._lib import lib
    from aotriton_amd.pyaotriton import T4
    B, H, Sq, Sk, causal = 1, 4, 300, 261, True
    q, k, v, _, do = make_inputs(B, H, H, Sq, Sk, D, BF, 'cuda', seed=16)
    b = torch.randn(B, H, Sq, Sk, device='cuda').to(BF)
    seed, off = (torch.tensor([x], device='cuda', dtype=torch.uint64) for x in (7, 8))
    null, sm, out = torch.empty([0], device='cuda', dtype=torch.uint64), 1 / math.sqrt(D), []
    o, L = torch.empty_like(q), torch.empty(B * H, Sq, device='cuda')
    assert flash.attn_fwd(q, k, v, b, sm, L, o, 0.2, seed, off, 0, null, null, None, causal, null) == flash.hipError_t.hipSuccess
    lib.fa_set_bwd_workspace_limit(-1 if stored else 0)
    try:
        for x in (b, b.transpose(2, 3).contiguous().transpose(2, 3)):
            grads = [torch.empty_like(t) for t in (q, k, v)]
            params = flash.fa_backward_op_params()
            flash._fill_bwd(params, q, k, v, None, sm, o, do, *grads, None, flash.lazy_dq_acc(q), L, flash.lazy_delta(L), 0.2,
                            seed, off, 0, causal)
            params.B = T4(x.data_ptr(), tuple(x.size()), x.stride(), flash.cast_dtype(BF))
            params.varlen_type = 0
            assert flash.fa_backward_op(params, params.kVersion, flash._stream(), None) == flash.hipError_t.hipSuccess
            out.append(grads)
    finally:
        lib.fa_set_bwd_workspace_limit(-1)
    for x, y in zip(*out):
        assert torch.isfinite(x).all() and torch.equal(x, y)


@pytest.mark.parametrize('D', [64, 128, 256])
@pytest.mark.parametrize('Sk', [136, 131])
def test_rows_that_a_bias_hides(D, Sk):
    """a finite bias that hides all keys of every other row: what stands for keys past the sequence must not reach dQ"""
    from aotriton_amd.autograd import attention
    q, k, v, b, do = make_inputs(4, 16, 16, 512, Sk, D, BF, 'cuda', seed=4, bias=True)
    b = b.contiguous()
    b[:, :, ::2] = -30000
    x = [t.clone().requires_grad_() for t in (q, k, v)]
    attention(*x, b, False, 1 / math.sqrt(D), 0.0)[0].backward(do)
    assert all(torch.isfinite(t.grad).all() for t in x)


@pytest.mark.parametrize('D', [64, 96, 128, 200, 256])
@pytest.mark.parametrize('Sk,dt,causal,p', [(136, BF, False, 0.0), (131, HF, False, 0.0), (264, HF, (150, 30), 0.0), (259, BF, True, 0.2), (136, HF, False, 0.2)])
def test_gradients_of_rows_that_a_bias_hides(D, Sk, dt, causal, p):
    """dS is stored.  A row's softmax does not change with a constant in its bias, so such rows have the gradients of a bias of zero; -256 is
    enough for what stands for keys past the sequence to overflow, and exact in 16 bits (it costs the exponents 2^-16)."""
    from aotriton_amd import flash
    from aotriton_amd.autograd import attention, AttentionExtraArgs
    from oracle import fa_ref
    from _util import FUDGE, check, keep_mask_from_oracle
    B, H, Sq = 1, 4, 300
    q, k, v, b, do = make_inputs(B, H, H, Sq, Sk, D, dt, 'cuda', seed=4, bias=True)
    b = b.contiguous()
    assert bwd(1, B, H, H, Sq, Sk, D, causal, p, bias=tuple(b.stride())).flags & 16
    hidden, zero = b.clone(), b.clone()
    hidden[:, :, ::2], zero[:, :, ::2] = -256, 0
    sm, ext = 1 / math.sqrt(D), AttentionExtraArgs(return_logsumexp=True, fillnan=True)
    x = [t.clone().requires_grad_() for t in (q, k, v)]
    attention(*x, hidden, causal, sm, p, ext)[0].backward(do)
    ct, wl, wr = flash.translate_causal(causal)
    keep = keep_mask_from_oracle(B, H, Sq, Sk, p, ext.philox_seed, ext.philox_offset1 + ext.philox_offset2, 'cuda')
    f = lambda t: t.float()
    ro, rl, _ = fa_ref.attn_fwd_ref(f(q), f(k), f(v), f(zero), sm, ct, wl, wr, p, keep)
    lo, ll, _ = fa_ref.attn_fwd_ref(q, k, v, zero, sm, ct, wl, wr, p, keep)
    rg = fa_ref.attn_bwd_ref(f(q), f(k), f(v), f(zero), sm, ro, f(do), rl, ct, wl, wr, p, keep)
    lg = fa_ref.attn_bwd_ref(q, k, v, zero, sm, lo, do, ll.to(dt).float().to(dt), ct, wl, wr, p, keep)
    for i, n in enumerate(('dq', 'dk', 'dv')):
        check(n, x[i].grad, rg[i], lg[i], FUDGE[n])
