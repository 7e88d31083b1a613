"""The forward's tile kernels without dropout, against the oracle.  Small calls go to the packed-rows kernel
(test_gpu_fwd_rows.py), so these have the heads that fill the chip: query rows and keys around the edges of the
tiles, masks that hide tiles and rows, a bias of every form; and tiles whose keys are split into parts.
test_launch_queries.py holds the cases to those kernels.  Tolerances are the reference's model (tests/_util.py)."""
import math

import pytest
import torch

from _util import FUDGE, LSE_ATOL, check, make_inputs

pytestmark = pytest.mark.gpu

BF, HF = torch.bfloat16, torch.float16
BR = (-2147483646, -2147483646)      # bottom right

TILES = [
    # B, Hq, Hk, Sq, Sk, D, dtype, causal, bias ('key': the same for all rows)
    (16, 32, 32, 256, 128, 64, BF, False, None),
    (16, 32, 8, 257, 129, 64, HF, True, None),
    (16, 32, 32, 411, 127, 64, BF, (60, -20), None),          # rows without a key
    (16, 32, 16, 513, 1, 64, HF, False, None),
    (16, 32, 32, 257, 300, 40, HF, BR, None),                 # head dim rounded up
    (16, 32, 32, 385, 63, 40, BF, False, None),
    (16, 32, 32, 256, 64, 128, HF, True, None),
    (16, 32, 32, 300, 160, 128, HF, False, None),
    (16, 32, 8, 300, 97, 128, BF, BR, None),
    (16, 32, 4, 511, 65, 128, BF, False, None),
    (16, 32, 32, 400, 200, 128, BF, (30, 90), None),
    (16, 32, 32, 257, 190, 96, HF, True, None),
    (16, 32, 32, 385, 130, 72, BF, BR, None),
    (16, 32, 32, 450, 100, 120, HF, False, None),
    (16, 32, 32, 128, 96, 256, BF, False, None),
    (16, 32, 16, 257, 161, 256, HF, True, None),
    (16, 32, 32, 200, 70, 200, BF, (25, 10), None),
    (16, 32, 32, 257, 140, 64, BF, False, 'full'),
    (16, 32, 8, 300, 97, 64, HF, True, 'full'),
    (16, 32, 32, 270, 130, 128, HF, (40, 40), 'full'),
    (16, 32, 32, 256, 90, 80, BF, False, 'full'),
    (16, 32, 32, 257, 66, 256, HF, True, 'full'),
    (16, 32, 32, 300, 384, 64, HF, False, 'key'),
    (16, 32, 16, 257, 131, 64, BF, True, 'key'),
    (16, 32, 32, 300, 333, 128, HF, (100, 30), 'key'),
    (16, 32, 32, 257, 93, 128, BF, False, 'key'),
    (16, 32, 32, 256, 200, 80, BF, True, 'key'),
    (16, 32, 32, 260, 77, 48, HF, False, 'key'),
]
SPLIT = [
    (1, 3, 1, 1025, 4097, 64, BF, False, None),
    (1, 3, 3, 1025, 4100, 48, HF, False, 'full'),
    (1, 8, 8, 2049, 2049, 64, HF, True, None),                # causal: parts without a tile
    (1, 8, 2, 2049, 2100, 64, BF, (2000, 100), 'full'),
    (1, 4, 4, 1025, 4097, 128, HF, False, None),
    (1, 4, 4, 1025, 4097, 96, BF, False, 'key'),              # (the parts take it as any bias)
    (1, 8, 8, 2049, 2200, 128, BF, BR, None),
    (1, 8, 4, 2200, 2049, 120, HF, BR, None),                 # the first rows see no key
    (1, 8, 4, 2049, 4097, 128, BF, (-300, 4000), None),       # the first keys are seen by no row
    (1, 4, 1, 1030, 4099, 128, BF, False, 'full'),
]


@pytest.mark.parametrize('case', TILES + SPLIT, ids=lambda c: '-'.join(str(x).replace('torch.', '') for x in c))
def test_forward_tiles_meet_the_oracle(case):
    from aotriton_amd import flash
    from aotriton_amd.autograd import attention, AttentionExtraArgs
    from oracle import fa_ref
    B, Hq, Hk, Sq, Sk, D, dtype, causal, bias = case
    q, k, v, b, _ = make_inputs(B, Hq, Hk, Sq, Sk, D, dtype, 'cuda', seed=51, bias=bias == 'full', bshd=True)
    if bias == 'key':
        g = torch.Generator(device='cpu').manual_seed(3)
        row = torch.randn(B, 1, 1, Sk, generator=g).to(dtype).to('cuda')
        b = row.masked_fill(torch.arange(Sk, device='cuda') >= (2 * Sk) // 3, float('-inf')).expand(B, Hq, Sq, Sk)
    sm = 1.0 / math.sqrt(D)
    o, _, L = attention(q, k, v, b, causal, sm, 0.0, AttentionExtraArgs(return_logsumexp=True, fillnan=True))
    torch.cuda.synchronize()
    ct, wl, wr = flash.translate_causal(causal)
    f = lambda t: None if t is None else t.float()
    ro, rl, _ = fa_ref.attn_fwd_ref(f(q), f(k), f(v), f(b), sm, ct, wl, wr)
    lo, _, _ = fa_ref.attn_fwd_ref(q, k, v, b, sm, ct, wl, wr)
    check('out', o, ro, lo, FUDGE['out'])
    L = L.view(B, Hq, Sq)
    assert torch.equal(torch.isinf(L), torch.isinf(rl))
    seen = torch.isfinite(rl)
    assert (L[seen] - rl[seen]).abs().max().item() <= LSE_ATOL
