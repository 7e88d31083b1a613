"""dK/dV of stored dS at head dims above 128 without a bias or with aligned rows of one: pairs of waves (fa_bwd_pair.h).  Against the oracle
where its steps and stages can go wrong: one step per q-head, fewer steps than stages, ragged tiles on both sides, windows, parts."""
import math

import pytest
import torch

from test_gpu_attention import _run_case
from test_launch_queries import bwd
from _util import make_inputs

pytestmark = pytest.mark.gpu

BF, HF = torch.bfloat16, torch.float16
CASES = [
    # B, Hq, Hk, Sq, Sk, D, Dv, dtype, causal, dropout, bias
    (2, 2, 2, 1, 1, 256, 256, BF, False, 0.0, False),              # one query, one key
    (1, 8, 2, 20, 136, 256, 256, HF, False, 0.0, False),           # one step per q-head, four heads to a kv-head
    (1, 6, 2, 33, 8, 256, 256, BF, False, 0.4, True),              # two steps per head, eight keys
    (2, 4, 4, 96, 128, 256, 256, HF, False, 0.1, True),            # as many steps as stages, a whole key tile
    (1, 4, 2, 97, 264, 256, 256, BF, True, 0.0, True),             # keys that no query sees
    (2, 2, 2, 300, 257, 256, 256, HF, True, 0.2, False),           # one key in the last tile
    (1, 2, 1, 515, 520, 256, 256, BF, (60, 90), 0.3, True),        # window: masked steps on both sides
    (1, 2, 2, 400, 400, 256, 256, HF, (150, -30), 0.0, True),
    (2, 4, 2, 260, 392, 136, 136, BF, True, 0.1, True),            # head dims rounded up
    (1, 4, 2, 129, 200, 200, 248, HF, False, 0.0, False),
    (1, 2, 2, 270, 264, 248, 160, BF, (40, 20), 0.2, True),
    (1, 8, 1, 700, 136, 256, 256, HF, True, 0.1, True),            # cut into parts
    (1, 2, 2, 1500, 130, 192, 192, BF, False, 0.0, False),
]


@pytest.mark.parametrize('case', CASES, ids=lambda c: '-'.join(str(x).replace('torch.', '') for x in c))
def test_pairs_meet_the_oracle(case):
    B, Hq, Hk, Sq, Sk, D, Dv, dtype, causal, p, bias = case
    x = bwd(1, B, Hq, Hk, Sq, Sk, max(D, Dv), causal, bias=bias, p=p)
    assert (x.block_m, x.block_n, x.num_waves) == (32, 128, 8) and x.flags & 16
    _run_case(B, Hq, Hk, Sq, Sk, D, dtype, causal, dropout_p=p, seed=17, Dv=Dv)
    if bias:
        _with_bias(B, Hq, Hk, Sq, Sk, D, Dv, dtype, causal, p)


def _with_bias(B, Hq, Hk, Sq, Sk, D, Dv, dtype, causal, p):
    """the bias without a gradient, so that small calls keep dS as well"""
    from aotriton_amd import flash
    from aotriton_amd.autograd import attention, AttentionExtraArgs
    from oracle import fa_ref
    from _util import FUDGE, check, keep_mask_from_oracle
    q, k, v, b, do = make_inputs(B, Hq, Hk, Sq, Sk, D, dtype, 'cuda', seed=18, bias=True, Dv=Dv)
    sm, ext = 1 / math.sqrt(D), AttentionExtraArgs(return_logsumexp=True, fillnan=True)
    x = [t.clone().requires_grad_() for t in (q, k, v)]
    attention(*x, b, causal, sm, p, ext)[0].backward(do)
    torch.cuda.synchronize()
    ct, wl, wr = flash.translate_causal(causal)
    keep = keep_mask_from_oracle(B, Hq, Sq, Sk, p, ext.philox_seed, ext.philox_offset1 + ext.philox_offset2, 'cuda')
    f = lambda t: t.float()
    ro, rl, _ = fa_ref.attn_fwd_ref(f(q), f(k), f(v), f(b), sm, ct, wl, wr, p, keep)
    lo, ll, _ = fa_ref.attn_fwd_ref(q, k, v, b, sm, ct, wl, wr, p, keep)
    rg = fa_ref.attn_bwd_ref(f(q), f(k), f(v), f(b), sm, ro, f(do), rl, ct, wl, wr, p, keep)
    lg = fa_ref.attn_bwd_ref(q, k, v, b, sm, lo, do, ll.to(dtype).float().to(dtype), ct, wl, wr, p, keep)
    for i, n in enumerate(('dq', 'dk', 'dv')):
        check(n, x[i].grad, rg[i], lg[i], FUDGE[n])
