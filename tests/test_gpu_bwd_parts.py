"""Backward with few key tiles and many queries or q-heads: the dK/dV items are cut into parts by q-heads
and by query tiles and a second kernel adds the parts up.  Against the oracle, at shapes where parts are
uneven, empty (masks) or end in ragged tiles, with and without stored dS."""
import math

import pytest
import torch

from test_gpu_attention import _run_case
from test_gpu_varlen_dropout import _run_varlen_case
from _util import make_inputs

pytestmark = pytest.mark.gpu

BF, HF = torch.bfloat16, torch.float16
CASES = [
    # B, Hq, Hk, Sq, Sk, D, dtype, causal, dropout, bias
    (1, 8, 2, 700, 100, 128, BF, False, 0.0, False),
    (1, 8, 1, 513, 129, 128, HF, True, 0.0, False),          # q-heads in parts; the second key tile has one key
    (1, 6, 2, 1500, 200, 128, BF, True, 0.0, False),         # three q-heads per group
    (2, 2, 2, 1100, 70, 128, BF, (60, 30), 0.0, False),      # window: parts without a tile
    (1, 4, 2, 900, 300, 64, HF, True, 0.0, False),
    (1, 4, 4, 1800, 250, 64, BF, False, 0.2, False),
    (1, 4, 1, 600, 150, 64, BF, False, 0.0, True),
    (1, 8, 2, 400, 190, 256, HF, True, 0.1, False),
    (1, 2, 2, 777, 65, 256, BF, False, 0.0, True),
    (1, 4, 2, 800, 100, 72, HF, False, 0.1, False),          # head dim rounded up
    (1, 4, 2, 500, 100, 113, BF, True, 0.0, False),          # through packed copies
    (1, 2, 2, 1500, 1400, 128, BF, True, 0.0, False),        # the last key tiles have fewer query tiles than parts
    (1, 2, 1, 1500, 1400, 64, HF, (700, 10), 0.0, False),
    (1, 2, 1, 1500, 700, 128, BF, (-200, 900), 0.1, False),  # keys that no row sees
]


@pytest.mark.parametrize('case', CASES, ids=lambda c: '-'.join(str(x).replace('torch.', '') for x in c))
def test_parts_meet_the_oracle(case, with_and_without_workspace):
    B, Hq, Hk, Sq, Sk, D, dtype, causal, p, bias = case
    if D == 113 and with_and_without_workspace != 'workspace':
        pytest.skip('element-wise kernels, which have no parts')
    _run_case(B, Hq, Hk, Sq, Sk, D, dtype, causal, dropout_p=p, bias=bias, seed=31)


@pytest.mark.parametrize('D', [64, 128])
def test_parts_of_packed_sequences(D):
    _run_varlen_case([700, 0, 33, 260], [90, 5, 300, 129], 8, 2, D, torch.bfloat16, True, 0, seed=5)


def test_parts_give_the_uncut_result():
    """the same call with the workspace limit at 0 (uncut, recomputing): equal up to summation order"""
    from aotriton_amd.autograd import attention
    from aotriton_amd._lib import lib
    q, k, v, _, do = make_inputs(1, 16, 2, 1000, 130, 64, torch.float16, 'cuda', seed=8)
    grads = []
    for limit in (-1, 0):
        lib.fa_set_bwd_workspace_limit(limit)
        x = [t.clone().requires_grad_() for t in (q, k, v)]
        attention(*x, None, True, 1 / math.sqrt(64), 0.0)[0].backward(do)
        torch.cuda.synchronize()
        grads.append([t.grad for t in x])
    lib.fa_set_bwd_workspace_limit(-1)
    for a, b in zip(*grads):
        # one rounding to fp16 (2^-11) of sums that differ in fp32 order
        assert ((a.float() - b.float()).abs() <= 2 ** -10 * b.float().abs() + 1e-4).all()
    assert torch.equal(grads[0][0], grads[1][0])      # dQ comes from the same kernel


@pytest.mark.parametrize('D', [128, 100])
def test_parts_give_way_to_the_stored_ds(D):
    """a limit that dS fits without the parts: dS is kept and the items run uncut (D 100: in the call on packed copies)"""
    from aotriton_amd.autograd import attention
    from aotriton_amd._lib import lib
    B, Hq, Hk, Sq, Sk = 1, 8, 2, 1500, 200
    up = lambda n: (n + 255) // 256 * 256
    tiles_q, tiles_k = (Sq + 63) // 64 | 1, (Sk + 127) // 128      # of 64 queries (an odd number of them) and 128 keys
    ds = B * Hq * tiles_q * tiles_k * 64 * 128 * 2 + 2 * up(B * Hq * Sq * 4)
    copies = 0 if D % 8 == 0 else 2 * (2 * up(B * Hq * Sq * 104 * 2) + 2 * up(B * Hk * Sk * 104 * 2))
    recomputed_differs = False
    for seed in range(9, 15):
        q, k, v, _, do = make_inputs(B, Hq, Hk, Sq, Sk, D, BF, 'cuda', seed=seed)
        dq = {}
        for limit in (-1, copies + ds, copies + ds - 256):
            lib.fa_set_bwd_workspace_limit(limit)
            x = [t.clone().requires_grad_() for t in (q, k, v)]
            attention(*x, None, False, 1 / math.sqrt(D), 0.0)[0].backward(do)
            torch.cuda.synchronize()
            dq[limit] = x[0].grad
        lib.fa_set_bwd_workspace_limit(-1)
        assert torch.equal(dq[copies + ds], dq[-1])
        # the recomputing kernel forms delta in another order: a few of the 1.5 million elements round the other way
        recomputed_differs |= not torch.equal(dq[copies + ds - 256], dq[-1])
        assert (dq[copies + ds - 256].float() - dq[-1].float()).abs().max() <= 2 ** -6 * dq[-1].float().abs().max()
    assert recomputed_differs
