"""dQ from stored dS at head dims 65-128 takes 64 keys a step with dB and where there are fewer workgroups than CUs, else 32: the same sums in
the same order, so the same bits, for steps that are whole, cut off by the last key, or seen by some rows only."""
import math

import pytest
import torch

from test_launch_queries import bwd
from _util import make_inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('D', [72, 96, 128])
@pytest.mark.parametrize('Sq, Sk, causal', [(100, 150, False), (130, 64, False), (257, 33, True), (90, 321, (40, 25)), (300, 8, False), (260, 200, True)])
@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16])
def test_both_steps_form_the_same_dq(D, Sq, Sk, causal, dtype):
    from aotriton_amd import flash
    H, sm = 4, 1 / math.sqrt(D)
    many = max(2 ** 22 // (H * Sq * Sk), 256 // H) + 1      # workgroups for every CU, pairs enough for dB from stored dS
    q, k, v, b, do = make_inputs(1, H, H, Sq, Sk, D, dtype, 'cuda', seed=12, bias=True)
    null, out = torch.empty([0], device='cuda', dtype=torch.uint64), []
    # one forward for all (a call of one batch element may take another kernel, whose O and logsumexp are rounded otherwise)
    w = b.contiguous()
    o0, L0 = torch.empty_like(q), torch.empty(H, Sq, device='cuda')
    assert flash.attn_fwd(q, k, v, w, sm, L0, o0, 0.0, null, null, 0, null, null, None, causal, null) == flash.hipError_t.hipSuccess
    for B, db in ((1, False), (many, False), (many, True)):
        assert bwd(2, B, H, H, Sq, Sk, D, causal, bias=True, db=db).flags & 16
        x, y, z, g, w, o = (t.expand(B, *t.shape[1:]).contiguous() for t in (q, k, v, do, b, o0))
        L = L0.expand(B, H, Sq).reshape(B * H, Sq)
        dq, dk, dv = (torch.full_like(t, float('nan')) for t in (x, y, z))
        dw = torch.empty_like(w) if db else None
        assert flash.attn_bwd(x, y, z, w, sm, o, g, dq, dk, dv, dw, flash.lazy_dq_acc(x), L, flash.lazy_delta(L), 0.0, null, null, 0,
                              causal) == flash.hipError_t.hipSuccess
        assert torch.isfinite(dq).all() and torch.equal(dq, dq[:1].expand_as(dq))
        out.append(dq[0])
    assert torch.equal(out[0], out[1]) and torch.equal(out[0], out[2])
