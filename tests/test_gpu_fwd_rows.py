"""The forward for few query rows per K/V head (fa_fwd_rows.h) against the oracle: blocks of 32 packed
rows around their edges, keys around the 32-key steps, the four waves' shares and the splits, masks that
leave splits, blocks or rows without a key.  Tolerances are the reference's model (tests/_util.py)."""
import math

import pytest
import torch

from _util import FUDGE, LSE_ATOL, check, make_inputs

pytestmark = pytest.mark.gpu

DEV = 'cuda'
BR = 2      # flash.CausalType.BOTTOM_RIGHT

CASES = [
    # B, Hq, Hk, Sq, Sk, D, dtype, causal, bias
    (1, 1, 1, 1, 1, 128, torch.bfloat16, False, False),
    (2, 4, 4, 1, 31, 64, torch.float16, False, False),
    (2, 8, 2, 1, 33, 128, torch.bfloat16, False, False),
    (1, 32, 8, 1, 2051, 128, torch.bfloat16, False, False),
    (3, 6, 2, 1, 127, 256, torch.float16, False, False),
    (1, 8, 1, 1, 4096, 256, torch.bfloat16, True, False),
    (1, 8, 2, 8, 129, 128, torch.float16, BR, False),           # one whole block of rows
    (2, 8, 2, 9, 1000, 128, torch.bfloat16, BR, False),         # a second block with four rows
    (1, 3, 1, 11, 513, 64, torch.bfloat16, BR, False),          # 33 rows
    (2, 2, 2, 63, 640, 64, torch.float16, True, False),         # top left: most keys hidden
    (1, 4, 2, 33, 300, 128, torch.float16, (20, 3), False),     # window: parts without a key
    (1, 4, 4, 40, 16, 128, torch.bfloat16, (4, -6), False),     # rows without a key
    (1, 4, 4, 64, 20, 128, torch.bfloat16, BR, False),          # bottom right with fewer keys than rows
    (2, 4, 4, 1, 200, 72, torch.bfloat16, False, False),        # head dim rounded up
    (1, 4, 2, 5, 777, 200, torch.float16, BR, False),
    (2, 4, 2, 3, 257, 128, torch.float16, False, True),
    (1, 8, 4, 7, 999, 64, torch.bfloat16, BR, True),
    (1, 2, 2, 16, 70, 256, torch.float16, (30, 30), True),
]


def _forward(q, k, v, b, sm, causal, split):
    """through the operator wrappers (scratch from torch's allocator) or, unsplit, without scratch"""
    from aotriton_amd import flash
    from aotriton_amd._lib import lib
    ok = flash.hipError_t.hipSuccess
    o = torch.full(q.shape[:3] + (v.shape[3],), float('nan'), device=DEV, dtype=q.dtype)
    L = torch.full((q.shape[0] * q.shape[1], q.shape[2]), float('nan'), device=DEV)
    null = torch.empty([0], device=DEV, dtype=torch.uint64)
    args = (q, k, v, b, sm, L, o, 0.0, null, null, 0, null, null, None, causal, null)
    if split == 'workspace':      # the C ABI without an allocator: the library's workspace
        assert flash.attn_fwd(*args, stream=flash._stream()) == ok
    elif split:
        assert flash.attn_fwd(*args) == ok
    else:
        lib.fa_set_bwd_workspace_limit(0)
        try:
            assert flash.attn_fwd(*args, stream=flash._stream()) == ok
        finally:
            lib.fa_set_bwd_workspace_limit(-1)
    torch.cuda.synchronize()
    return o, L


@pytest.mark.parametrize('case', CASES, ids=lambda c: '-'.join(str(x).replace('torch.', '') for x in c))
def test_few_rows_meet_the_oracle(case):
    from aotriton_amd import flash
    from oracle import fa_ref
    B, Hq, Hk, Sq, Sk, D, dtype, causal, bias = case
    q, k, v, b, _ = make_inputs(B, Hq, Hk, Sq, Sk, D, dtype, DEV, seed=21, bias=bias, bshd=True)
    if causal == BR:
        causal = flash.CausalType.BOTTOM_RIGHT
    sm = 1.0 / math.sqrt(D)
    ct, wl, wr = flash.translate_causal(causal)
    f = lambda t: None if t is None else t.float()
    ro, rl, _ = fa_ref.attn_fwd_ref(f(q), f(k), f(v), f(b), sm, ct, wl, wr)
    lo, _, _ = fa_ref.attn_fwd_ref(q, k, v, b, sm, ct, wl, wr)
    for split in (True, 'workspace', False):
        o, L = _forward(q, k, v, b, sm, causal, split)
        check('out', o, ro, lo, FUDGE['out'])
        L = L.view(B, Hq, Sq)
        assert torch.equal(torch.isinf(L), torch.isinf(rl))
        seen = torch.isfinite(rl)
        assert (L[seen] - rl[seen]).abs().max().item() <= LSE_ATOL if seen.any() else True


def _scratch_bytes(rows, D):      # the parts' fp32 sums and statistics
    return rows * (4 * D + 8)


def _scratch_of(call):
    """its result, and the memory that it held beside its result: the scratch of a split forward (_forward's outputs excluded)"""
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    out = call()
    stats = torch.cuda.memory_stats()
    return out, stats['requested_bytes.all.peak'] - stats['requested_bytes.all.current']


@pytest.mark.parametrize('D', [64, 128, 256])
@pytest.mark.parametrize('parts', [2, 3, 4, 5, 8, 9, 17, 63, 64])
def test_sums_of_few_and_many_parts(parts, D):
    """One row block and 128 keys a part (four waves of 32): up to eight parts each thread has all of its columns' (two, or two
    groups of four), beyond that the threads of a workgroup share them.  (Two parts of that many keys do not pay; of 1024 and for
    100 K/V heads they do.)"""
    from oracle import fa_ref
    Hk, Sk = (100, 1024) if parts == 2 else (1, 128 * parts)
    q, k, v, _, _ = make_inputs(1, 5 * Hk, Hk, 1, Sk, D, torch.bfloat16, DEV, seed=parts)
    f = lambda t: t.float()
    sm = D ** -0.5
    ro, rl, _ = fa_ref.attn_fwd_ref(f(q), f(k), f(v), None, sm, 0, 0, 0)
    lo, _, _ = fa_ref.attn_fwd_ref(q, k, v, None, sm, 0, 0, 0)
    (o, L), scratch = _scratch_of(lambda: _forward(q, k, v, None, sm, False, True))
    assert scratch == _scratch_bytes(parts * 5 * Hk, D)      # as many parts of five rows
    check('out', o, ro, lo, FUDGE['out'])
    assert (L.view(1, 5 * Hk, 1) - rl).abs().max().item() <= LSE_ATOL


@pytest.mark.parametrize('D, H, Sq, Sk, parts', [
    (64, 8, 767, 3000, 5), (64, 5, 1000, 3000, 8), (64, 4, 767, 4100, 9), (64, 2, 1030, 8192, 10), (64, 4, 1000, 11825, 16),
    (128, 5, 1000, 4100, 5), (128, 5, 1000, 6000, 8), (128, 4, 1000, 11825, 9), (128, 4, 767, 6000, 12), (128, 2, 1030, 11825, 15)])
def test_sums_of_many_parts_of_many_rows(D, H, Sq, Sk, parts):
    """split tiles have more rows than packed rows ever do: all parts of a column in one thread, in two to four groups of four"""
    from oracle import fa_ref
    q, k, v, _, _ = make_inputs(1, H, H, Sq, Sk, D, torch.bfloat16, DEV, seed=parts)
    f = lambda t: t.float()
    sm = D ** -0.5
    ro, rl, _ = fa_ref.attn_fwd_ref(f(q), f(k), f(v), None, sm, 0, 0, 0)
    lo, _, _ = fa_ref.attn_fwd_ref(q, k, v, None, sm, 0, 0, 0)
    (o, L), scratch = _scratch_of(lambda: _forward(q, k, v, None, sm, False, True))
    assert scratch == _scratch_bytes(parts * H * ((Sq + 255) // 256) * 256, D)
    check('out', o, ro, lo, FUDGE['out'])
    assert (L.view(1, H, Sq) - rl).abs().max().item() <= LSE_ATOL


def test_scores_that_grow_and_huge_scores():
    """the reference maximum moves in every step of every wave, and 16-bit scores of 1e4"""
    from oracle import fa_ref
    q, k, v, _, _ = make_inputs(1, 4, 2, 2, 900, 128, torch.bfloat16, DEV, seed=4)
    k = k * torch.linspace(0.1, 60.0, 900, device=DEV, dtype=torch.float32).to(k.dtype).view(1, 1, -1, 1)
    f = lambda t: t.float()
    ro, rl, _ = fa_ref.attn_fwd_ref(f(q), f(k), f(v), None, 0.3, 0, 0, 0)
    lo, _, _ = fa_ref.attn_fwd_ref(q, k, v, None, 0.3, 0, 0, 0)
    o, L = _forward(q, k, v, None, 0.3, False, True)
    check('out', o, ro, lo, FUDGE['out'])
    assert ((L.view(1, 4, 2) - rl).abs() <= 1e-5 * rl.abs() + LSE_ATOL).all()


def test_packed_decode_batch():
    """one query per packed sequence, caches of different lengths (one of them empty)"""
    from aotriton_amd.autograd import attention_varlen, AttentionExtraArgs
    from oracle import fa_ref
    lk = [700, 1, 0, 64, 333]
    n, Hq, Hk, D = len(lk), 8, 2, 128
    g = torch.Generator().manual_seed(2)
    mk = lambda H, T: torch.randn(1, T, H, D, generator=g).to(torch.float16).to(DEV).transpose(1, 2)
    q, k, v = mk(Hq, n), mk(Hk, sum(lk)), mk(Hk, sum(lk))
    o, _, L = attention_varlen(q, k, v, [1] * n, lk, False, 0.1, 0.0, AttentionExtraArgs(return_logsumexp=True, fillnan=True))
    at = 0
    for i, len_k in enumerate(lk):
        if len_k == 0:
            assert (o[:, :, i] == 0).all() and torch.isinf(L[:, i]).all()
            continue
        ks, vs = k[:, :, at:at + len_k], v[:, :, at:at + len_k]
        ro, rl, _ = fa_ref.attn_fwd_ref(q[:, :, i:i + 1].float(), ks.float(), vs.float(), None, 0.1, 0, 0, 0)
        lo, _, _ = fa_ref.attn_fwd_ref(q[:, :, i:i + 1], ks, vs, None, 0.1, 0, 0, 0)
        check('out', o[:, :, i:i + 1], ro, lo, FUDGE['out'])
        assert (L[:, i] - rl.view(-1)).abs().max().item() <= LSE_ATOL
        at += len_k


def test_split_forward_replays_from_a_hip_graph():
    """scratch under capture is the graph's own: replays, with eager calls between them, repeat the eager bits"""
    from aotriton_amd.torch_ops import scaled_dot_product_attention as sdpa
    q, k, v, _, _ = make_inputs(2, 8, 2, 1, 1500, 128, torch.bfloat16, DEV, seed=6)
    run = lambda: sdpa(q, k, v, enable_gqa=True)
    eager = run().clone()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        run()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        captured = run()
    for _ in range(3):
        captured.fill_(float('nan'))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(captured, eager)
        assert torch.equal(run(), eager)


@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float32])
def test_logsumexp_where_waves_meet(dtype):
    """L = (m sc + log2 l) ln 2 with m sc never rounded by itself.  For these rows m sc lies around 4.6 and the sum in
    [8, 16): its rounding (2^-20 wide, rms 2.8e-7) times ln 2, that of the product (2^-21, 1.4e-7) and half as much
    from the scores and the logarithm make 4.1e-8 of L; a rounded m sc (2^-21) makes it 4.5e-8."""
    from aotriton_amd.autograd import attention, AttentionExtraArgs
    B, Hq, Hk, Sk, D = 8, 32, 8, 700, 128
    err, n = 0.0, 10
    for seed in range(n):
        g = torch.Generator(device=DEV).manual_seed(seed)
        q, k = (torch.randn(B, h, s, D, device=DEV, generator=g).to(dtype) for h, s in ((Hq, 1), (Hk, Sk)))
        _, _, L = attention(q, k, k, None, False, D ** -0.5, 0.0, AttentionExtraArgs(return_logsumexp=True))
        kt = k.double().repeat_interleave(Hq // Hk, 1).transpose(-1, -2).contiguous()
        want = torch.logsumexp(torch.matmul(q.double(), kt) * D ** -0.5, -1).reshape(L.shape)
        err += ((L.double() - want).norm() / want.norm()).item() / n
    assert err < 4.3e-8
