"""Forward tiles of 128 rows with three workgroups per CU (head dims up to 64), and those and two per CU under a bias of the
keys: at ragged last tiles and the fewest keys, against a computation in 64 bits."""
import pytest
import torch

from test_gpu_attention import _run_case
from test_launch_queries import fwd

BF, HF = torch.bfloat16, torch.float16
THREE = [
    # B, Hq, Hk, Sq, Sk, D, dtype, causal
    (40, 16, 16, 128, 1, 64, BF, False),
    (16, 32, 8, 325, 325, 64, HF, True),
    (16, 12, 12, 384, 33, 64, BF, False),
    (16, 32, 32, 257, 129, 64, HF, True),
    (16, 32, 32, 257, 161, 48, BF, (-2147483646, -2147483646)),
    (16, 12, 12, 383, 300, 40, HF, False),
]
# a boolean mask of the keys, as the SDPA entry point passes it on
KEYS = [
    (16, 12, 384, 384, 64, HF),
    (16, 32, 130, 65, 64, BF),
    (40, 16, 128, 97, 40, HF),
    (16, 36, 290, 131, 128, BF),
    (16, 36, 290, 31, 80, HF),
]


def _id(c):
    return '-'.join(str(x).replace('torch.', '') for x in c)


def test_cases_are_of_these_tiles():
    for c in THREE:
        assert (lambda x: (x.block_m, x.block_n, x.num_waves))(fwd(*c[:6], c[7])) == (128, 32, 4), _id(c)
    assert fwd(8, 32, 32, 1369, 1369, 64, True).block_m == 256 and fwd(64, 32, 32, 300, 300, 64).block_m == 256


@pytest.mark.gpu
@pytest.mark.parametrize('case', THREE, ids=_id)
def test_three_per_cu_meet_the_oracle(case):
    _run_case(*case, seed=29)


@pytest.mark.gpu
@pytest.mark.parametrize('case', KEYS, ids=_id)
def test_key_masks(case):
    from aotriton_amd import sdpa
    B, H, Sq, Sk, D, dt = case
    g = torch.Generator(device='cuda').manual_seed(3)
    q, k, v = (torch.randn(B, H, s, D, device='cuda', generator=g).to(dt) for s in (Sq, Sk, Sk))
    mask = torch.rand(B, 1, 1, Sk, device='cuda', generator=g) < 0.7
    mask[..., 0] = True
    o = sdpa.scaled_dot_product_attention(q, k, v, attn_mask=mask)
    s = torch.matmul(q.double(), k.double().transpose(-1, -2).contiguous()) * D ** -0.5
    p = torch.softmax(s.masked_fill(~mask, float('-inf')), -1)
    want = torch.matmul(p, v.double())
    # P rounded to the 16-bit type, the fp32 sums, the result rounded: 3 roundings of the type in the norm
    assert ((o.double() - want).norm() / want.norm()).item() < 3 * torch.finfo(dt).eps / 2


BOOL = KEYS + [
    (1, 16, 1, 3000, 64, BF),              # packed rows, split keys
    (4, 16, 142, 142, 80, HF),             # packed rows
    (2, 16, 7, 70, 128, BF),
    (16, 32, 300, 300, 128, HF),           # whole tiles
    (40, 32, 520, 200, 64, BF),
    (1, 4, 1030, 4099, 128, BF),           # split tiles, other head dims and types: the mask is made additive first
    (2, 8, 200, 96, 256, BF),
    (2, 4, 60, 50, 64, torch.float32),
    (2, 4, 60, 50, 36, HF),
]


@pytest.mark.gpu
@pytest.mark.parametrize('form', ['batch', 'head', 'one', 'vector', 'strided', 'one key', 'hidden'])
@pytest.mark.parametrize('case', BOOL, ids=_id)
def test_boolean_key_masks_are_the_additive_ones(case, form):
    """To the bit: the forward reads the boolean mask as 0 and -inf."""
    from aotriton_amd.torch_ops import scaled_dot_product_attention as sdpa
    B, H, Sq, Sk, D, dt = case
    g = torch.Generator(device='cuda').manual_seed(5)
    q, k, v = (torch.randn(B, H, s, D, device='cuda', generator=g).to(dt) for s in (Sq, Sk, Sk))
    shape = {'batch': (B, 1, 1, Sk), 'head': (B, H, 1, Sk), 'one': (1, 1, 1, Sk), 'vector': (Sk,), 'strided': (B, 1, 1, 3 * Sk),
             'one key': (B, 1, 1, 1), 'hidden': (B, 1, 1, Sk)}[form]
    mask = torch.rand(shape, device='cuda', generator=g) < 0.7
    if form == 'strided':
        mask = mask[..., 1::3]
    if form == 'hidden':      # (an element of the batch without a key: zeros)
        mask[B - 1] = False
    additive = torch.zeros(mask.shape, device='cuda', dtype=dt).masked_fill(~mask, float('-inf'))
    assert torch.equal(sdpa(q, k, v, attn_mask=mask), sdpa(q, k, v, attn_mask=additive))
    # the route that keeps what the backward needs takes the additive mask
    qg = q.clone().requires_grad_()
    og = sdpa(qg, k, v, attn_mask=mask)
    assert og.requires_grad and torch.equal(og, sdpa(q, k, v, attn_mask=additive))


GROUPED = [      # B, Hq, Hk, Sq, Sk, D, dtype, packed rows?
    (1, 32, 8, 1, 3000, 128, BF, True),
    (2, 12, 4, 7, 501, 64, HF, True),
    (3, 6, 2, 11, 401, 40, BF, True),
    (16, 16, 4, 300, 301, 64, HF, False),
    (8, 32, 8, 290, 131, 128, BF, False),
]
TL, BOTTOM_RIGHT = -2147483647, -2147483646


@pytest.mark.gpu
@pytest.mark.parametrize('case', GROUPED, ids=_id)
def test_boolean_key_masks_per_head_with_fewer_kv_heads(case):
    """a mask of its own for every query head, whose rows are packed by K/V head in one of the kernels: the additive one's bits"""
    from aotriton_amd.torch_ops import scaled_dot_product_attention as sdpa
    B, Hq, Hk, Sq, Sk, D, dt, rows = case
    assert bool(fwd(B, Hq, Hk, Sq, Sk, D, bias=True).flags & 128) == rows
    g = torch.Generator(device='cuda').manual_seed(5)
    q, k, v = (torch.randn(B, h, s, D, device='cuda', generator=g).to(dt) for h, s in ((Hq, Sq), (Hk, Sk), (Hk, Sk)))
    for shape in ((B, Hq, 1, Sk), (1, Hq, 1, Sk), (B, 1, 1, Sk)):
        mask = torch.rand(shape, device='cuda', generator=g) < 0.7
        additive = torch.zeros(shape, device='cuda', dtype=dt).masked_fill(~mask, float('-inf'))
        assert torch.equal(sdpa(q, k, v, attn_mask=mask, enable_gqa=True), sdpa(q, k, v, attn_mask=additive, enable_gqa=True))


@pytest.mark.gpu
@pytest.mark.parametrize('window', [(0, 0, 0), (3, TL, TL), (3, BOTTOM_RIGHT, BOTTOM_RIGHT), (3, 40, 25), (3, 100, -3)])
@pytest.mark.parametrize('case', GROUPED, ids=_id)
def test_key_mask_entry_point_takes_windows(case, window):
    """fa_attn_fwd_key_mask against fa_attn_fwd with the additive mask, under every kind of window: the same bits; rows of a mask
    and other element types are refused"""
    import ctypes
    from aotriton_amd._lib import lib
    from aotriton_amd.flash import mk_aotensor
    from aotriton_amd.pyaotriton.v3.flash import attn_fwd_params
    B, Hq, Hk, Sq, Sk, D, dt, _ = case
    g = torch.Generator(device='cuda').manual_seed(5)
    q, k, v = (torch.randn(B, h, s, D, device='cuda', generator=g).to(dt) for h, s in ((Hq, Sq), (Hk, Sk), (Hk, Sk)))
    mask = torch.rand(B, Hq, 1, Sk, device='cuda', generator=g) < 0.7
    additive = torch.zeros(mask.shape, device='cuda', dtype=dt).masked_fill(~mask, float('-inf'))
    stream, out = torch.cuda.current_stream().cuda_stream, []
    for b in (mask.view(torch.uint8), additive):
        o, L = torch.full_like(q, 7.0), torch.full((B * Hq, Sq), 7.0, device='cuda')
        x = attn_fwd_params()
        x.Q, x.K, x.V, x.Out, x.L, x.B = (mk_aotensor(t) for t in (q, k, v, o, L, b.expand(B, Hq, Sq, Sk)))
        x.Sm_scale, x.causal_type, x.window_left, x.window_right = D ** -0.5, *window
        c = x.to_c()
        if b is additive:
            rc = lib.fa_attn_fwd(ctypes.byref(c), x.kVersion, stream, None)
            assert lib.fa_attn_fwd_key_mask(ctypes.byref(c), x.kVersion, stream, None, None) == 1      # not a mask of bytes
        else:
            rc = lib.fa_attn_fwd_key_mask(ctypes.byref(c), x.kVersion, stream, None, None)
            if Sq > 1:
                c.B.strides[2] = Sk
                assert lib.fa_attn_fwd_key_mask(ctypes.byref(c), x.kVersion, stream, None, None) == 801
        assert rc == 0
        out.append((o, L))
    assert torch.equal(out[0][0], out[1][0]) and torch.equal(out[0][1], out[1][1])


@pytest.mark.gpu
@pytest.mark.parametrize('score', ['inf', '-inf', 'nan'])
@pytest.mark.parametrize('case', [(1, 16, 1, 3000, 64, BF), (2, 16, 7, 70, 128, HF), (16, 12, 384, 384, 64, HF)], ids=_id)
def test_hidden_keys_of_any_score(case, score):
    """a hidden key whose score is infinite or NaN: in the packed-rows kernel as in the tiles what the additive mask gives"""
    from aotriton_amd.torch_ops import scaled_dot_product_attention as sdpa
    B, H, Sq, Sk, D, dt = case
    g = torch.Generator(device='cuda').manual_seed(5)
    q, k, v = (torch.randn(B, H, s, D, device='cuda', generator=g).to(dt) for s in (Sq, Sk, Sk))
    q[..., 0] = 1.0
    k[0, 3, 17] = 0.0
    k[0, 3, 17, 0] = float(score)      # one key of one head
    mask = torch.ones(B, 1, 1, Sk, device='cuda', dtype=torch.bool)
    mask[..., 17] = False
    additive = torch.zeros(mask.shape, device='cuda', dtype=dt).masked_fill(~mask, float('-inf'))
    o, want = sdpa(q, k, v, attn_mask=mask), sdpa(q, k, v, attn_mask=additive)
    assert torch.equal(o.isnan(), want.isnan()) and torch.equal(o.nan_to_num(), want.nan_to_num())
    assert want[0, 3].isnan().any().item() == (score != '-inf')


@pytest.mark.gpu
@pytest.mark.parametrize('case', BOOL[-4:], ids=_id)
def test_masks_made_additive_cost_one_allocation(case):
    """a boolean mask that the kernels do not read: its additive copy, the outputs, and nothing twice"""
    from aotriton_amd.torch_ops import scaled_dot_product_attention as sdpa
    B, H, Sq, Sk, D, dt = case
    q, k, v = (torch.randn(B, H, s, D, device='cuda').to(dt) for s in (Sq, Sk, Sk))
    mask = torch.rand(B, 1, 1, Sk, device='cuda') < 0.7
    additive = torch.zeros(mask.shape, device='cuda', dtype=dt).masked_fill(~mask, float('-inf'))
    count = lambda: torch.cuda.memory_stats()['allocation.all.allocated']
    taken = []
    for m in (mask, additive):
        sdpa(q, k, v, attn_mask=m)
        before = count()
        sdpa(q, k, v, attn_mask=m)
        taken.append(count() - before)
    assert taken[0] == taken[1] + 1


def test_fake_key_mask_op():
    import aotriton_amd.torch_ops  # noqa: F401
    q = torch.empty(2, 4, 8, 64, device='meta', dtype=HF)
    o, lse = torch.ops.aotriton_amd.flash_attention_forward_key_mask(q, q, q, torch.empty(2, 1, 1, 8, device='meta', dtype=torch.bool), 1.0)
    assert o.shape == q.shape and lse.shape == (8, 8)
