"""Backward with 64 rows per wave (256-row workgroups): against the oracle, and against the 128-row kernels on a part of the
batch too small for it, at the edges of its tiles: 32-row steps, 64-row waves, 256-row items, windows that leave waves
without work, three and fewer steps (the depth of its staging), head dims rounded up."""
import math

import numpy as np
import pytest
import torch

from test_gpu_attention import _run_case
from test_gpu_varlen_dropout import _run_varlen_case
from test_launch_queries import bwd, packed
from _util import make_inputs

BF, HF = torch.bfloat16, torch.float16
CASES = [
    # B, Hq, Hk, Sq, Sk, D, dtype, causal, bshd
    (16, 16, 16, 257, 257, 128, BF, True, False),            # a second item of one row
    (16, 16, 16, 321, 256, 128, HF, False, True),
    (16, 16, 16, 192, 320, 128, BF, True, False),            # keys that no query sees
    (32, 16, 8, 223, 223, 128, BF, True, True),              # two q-heads per kv-head
    (16, 16, 16, 290, 290, 128, BF, (0, 0), False),          # one visible key per query
    (16, 16, 16, 300, 447, 128, HF, (100, 20), False),
    (16, 16, 16, 310, 310, 128, BF, (-90, 200), False),      # rows without a key, waves without a visible tile
    (16, 16, 16, 190, 380, 96, BF, True, False),
    (16, 16, 16, 383, 190, 72, HF, False, True),
    (16, 16, 16, 255, 255, 112, BF, True, False),
]


def _id(c):
    return '-'.join(str(x).replace('torch.', '') for x in c)


def test_cases_are_of_these_kernels():
    for case in CASES:
        c1, c2 = (bwd(slot, *case[:6], case[7]) for slot in (1, 2))
        assert (c1.block_m, c1.block_n) == (32, 256) or (c2.block_m, c2.block_n) == (256, 32), _id(case)
    for case in CASES[:1] + CASES[7:8]:
        assert bwd(1, *case[:6], case[7]).block_n == 256 and bwd(2, *case[:6], case[7]).block_m == 256
    assert bwd(1, 1, 8, 8, 1024, 1024, 128).block_n == 128      # too few items
    assert bwd(2, 16, 16, 16, 257, 257, 128, True, p=0.1).block_m == 128 and bwd(2, 16, 16, 16, 257, 257, 64, True).block_m == 128


@pytest.mark.gpu
@pytest.mark.parametrize('case', CASES, ids=_id)
def test_wide_items_meet_the_oracle(case):
    B, Hq, Hk, Sq, Sk, D, dtype, causal, bshd = case
    from aotriton_amd._lib import lib
    lib.fa_set_bwd_workspace_limit(0)      # (so that each kernel runs wherever the rule takes it, also without the other)
    try:
        _run_case(B, Hq, Hk, Sq, Sk, D, dtype, causal, seed=17, bshd=bshd)
    finally:
        lib.fa_set_bwd_workspace_limit(-1)


@pytest.mark.gpu
@pytest.mark.parametrize('causal', [False, True, (70, 9)])
def test_wide_items_give_the_result_of_narrow_ones(causal):
    """the same products summed in the same order: equal bits"""
    from aotriton_amd import flash
    from aotriton_amd._lib import lib
    ok = flash.hipError_t.hipSuccess
    S, sm = 330, 1 / math.sqrt(128)
    q, k, v, _, do = make_inputs(16, 16, 16, S, S, 128, BF, 'cuda', seed=4)
    assert bwd(1, 16, 16, 16, S, S, 128, causal).block_n == 256 and bwd(1, 1, 16, 16, S, S, 128, causal).block_n == 128
    o, lse = torch.empty_like(q), torch.empty(16 * 16, S, device='cuda')
    none, counter = torch.empty(0, device='cuda', dtype=torch.uint64), torch.zeros(1, device='cuda', dtype=torch.int32)
    assert flash.attn_fwd(q, k, v, None, sm, lse, o, 0.0, none, none, 0, none, none, None, causal, counter) == ok
    lib.fa_set_bwd_workspace_limit(0)
    grads = []
    try:
        for n in (16, 1):
            g = [torch.empty_like(t[:n]) for t in (q, k, v)]
            lse_n = lse[:16 * n]
            assert flash.attn_bwd(q[:n], k[:n], v[:n], None, sm, o[:n], do[:n], *g, None, None, lse_n,
                                  torch.empty_like(lse_n), 0.0, none, none, 0, causal) == ok
            torch.cuda.synchronize()
            grads.append([t[:1] for t in g])
    finally:
        lib.fa_set_bwd_workspace_limit(-1)
    for a, b in zip(*grads):
        assert torch.equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize('D, causal', [(128, True), (96, False), (128, (50, 30))])
def test_wide_items_of_packed_sequences(D, causal):
    lens = np.random.default_rng(3).integers(100, 500, size=24)
    lens[5], lens[11] = 0, 257
    _run_varlen_case(lens, lens[::-1].copy() if D == 96 else lens, 16, 16, D, BF, causal, 0, seed=6)


PACKED = np.random.default_rng(3).integers(100, 500, size=24) * 2 + 1
PACKED[5], PACKED[11], PACKED[17] = 0, 257, 1
PACKED_CASES = [(128, True, 16, 16), (128, (50, 30), 16, 16), (96, False, 16, 16), (72, True, 64, 32), (128, (-40, 200), 32, 32)]


def test_packed_cases_are_of_these_kernels():
    for D, causal, Hq, Hk in PACKED_CASES:
        c1, c2 = (packed(slot, PACKED, PACKED[::-1] if D == 96 else PACKED, Hq, Hk, D, causal) for slot in (1, 2))
        assert (c1.block_m, c1.block_n, c2.block_m, c2.block_n) == (32, 256, 256, 32), (D, causal, Hq, Hk)


@pytest.mark.gpu
@pytest.mark.parametrize('D, causal, Hq, Hk', PACKED_CASES)
def test_packed_sequences_on_both_kernels_meet_the_oracle(D, causal, Hq, Hk):
    _run_varlen_case(PACKED, PACKED[::-1].copy() if D == 96 else PACKED, Hq, Hk, D, HF if D == 72 else BF, causal, 0, seed=16)
