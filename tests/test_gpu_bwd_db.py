"""dB written by the kernel that forms dQ from the stored dS: against the oracle at the edges of its steps and
tiles, rows and tiles no key of which is visible, and rows whose end is no whole 16-byte piece."""
import math

import pytest
import torch

from test_gpu_attention import _run_case
from _util import make_inputs

pytestmark = pytest.mark.gpu

BF, HF = torch.bfloat16, torch.float16
CASES = [
    # B, Hq, Hk, Sq, Sk, D, dtype, causal, dropout
    (20, 12, 12, 130, 136, 64, BF, False, 0.0),
    (4, 16, 4, 300, 264, 64, HF, True, 0.0),
    (3, 14, 14, 520, 200, 64, BF, (40, 10), 0.1),       # most rows see no key; dropout takes the narrow stored tiles
    (10, 12, 12, 70, 600, 128, HF, True, 0.0),          # key tiles that no row sees
    (4, 16, 8, 257, 328, 128, BF, (100, -3), 0.0),
    (30, 20, 20, 100, 72, 80, HF, False, 0.1),
    (160, 100, 100, 33, 8, 40, BF, False, 0.0),
    (4, 14, 14, 290, 296, 256, HF, True, 0.1),
    (20, 20, 20, 65, 168, 200, BF, (20, 20), 0.0),
    (2, 4, 4, 256, 256, 64, HF, True, 0.0),             # below the line: recomputed
]


@pytest.mark.parametrize('case', CASES, ids=lambda c: '-'.join(str(x).replace('torch.', '') for x in c))
def test_db_meets_the_oracle(case):
    B, Hq, Hk, Sq, Sk, D, dtype, causal, p = case
    _run_case(B, Hq, Hk, Sq, Sk, D, dtype, causal, dropout_p=p, bias=True, seed=41)


@pytest.mark.parametrize('Sk', [9, 61, 131, 190])
@pytest.mark.parametrize('D', [64, 128, 256])
def test_db_rows_with_a_ragged_end(Sk, D):
    """dB as a view of wider rows: the result of the recomputing backward, and nothing written past the rows' end"""
    from aotriton_amd import flash
    from aotriton_amd._lib import lib
    H, Sq = 64, 300
    B = 2 ** 22 // (H * Sq * Sk) + 1      # large enough for the stored dS
    q, k, v, _, do = make_inputs(B, H, H, Sq, Sk, D, HF, 'cuda', seed=6)
    wide = (Sk + 7) // 8 * 8 + 8
    b = torch.randn(B, H, Sq, wide, device='cuda', dtype=HF)[..., :Sk]
    sm, null = 1 / math.sqrt(D), torch.empty([0], device='cuda', dtype=torch.uint64)
    o, L = torch.empty_like(q), torch.empty(B * H, Sq, device='cuda')
    assert flash.attn_fwd(q, k, v, b, sm, L, o, 0.0, null, null, 0, null, null, None, True, null) == flash.hipError_t.hipSuccess
    out = []
    for limit in (-1, 0):
        lib.fa_set_bwd_workspace_limit(limit)
        full = torch.full((B, H, Sq, wide), 7.0, device='cuda', dtype=HF)
        dq, dk, dv = torch.empty_like(q), torch.empty_like(k), torch.empty_like(v)
        err = flash.attn_bwd(q, k, v, b, sm, o, do, dq, dk, dv, full[..., :Sk], flash.lazy_dq_acc(q), L,
                             flash.lazy_delta(L), 0.0, null, null, 0, True)
        torch.cuda.synchronize()
        lib.fa_set_bwd_workspace_limit(-1)
        assert err == flash.hipError_t.hipSuccess
        assert (full[..., Sk:] == 7.0).all()
        out.append((full[..., :Sk].float(), dq.float()))
    # dP and delta are fp32 sums of D products of size <= 4 sqrt(D) together, in another order (D 2^-24 of that); then both round to fp16, dS before dQ is summed
    sums = D * 2 ** -24 * 4 * math.sqrt(D)
    for x, y in zip(*out):
        assert ((x - y).abs() <= 2 ** -9 * y.abs() + 2e-3 * y.abs().max() + sums).all()
