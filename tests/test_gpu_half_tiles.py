"""Forward tiles of 128 rows, two workgroups per CU, where 256-row tiles leave rounds empty: many heads with
sequences a little over half a tile or a tile.  Against the oracle at ragged last tiles, masks and dropout."""
import pytest
import torch

from test_gpu_attention import _run_case

pytestmark = pytest.mark.gpu

BF, HF = torch.bfloat16, torch.float16
CASES = [
    # B, Hq, Hk, Sq, Sk, D, dtype, causal, dropout
    (40, 16, 16, 128, 128, 64, BF, False, 0.0),       # 3 rounds against 2
    (40, 16, 4, 97, 130, 64, HF, True, 0.1),
    (20, 32, 32, 1, 300, 64, BF, False, 0.1),         # (without dropout the rows kernel takes it)
    (40, 16, 8, 113, 65, 128, BF, (40, 9), 0.0),
    (16, 36, 36, 129, 33, 128, HF, False, 0.2),
    (40, 16, 16, 128, 97, 96, HF, True, 0.0),
    (40, 16, 16, 70, 128, 40, BF, False, 0.0),
    (40, 16, 16, 70, 128, 40, BF, False, 0.1),        # (without dropout the rows kernel takes it)
    (16, 36, 36, 290, 33, 128, HF, False, 0.2),       # 5 rounds against 4, a ragged third tile
]


@pytest.mark.parametrize('case', CASES, ids=lambda c: '-'.join(str(x).replace('torch.', '') for x in c))
def test_half_tiles_meet_the_oracle(case):
    B, Hq, Hk, Sq, Sk, D, dtype, causal, p = case
    _run_case(B, Hq, Hk, Sq, Sk, D, dtype, causal, dropout_p=p, seed=23)


@pytest.mark.parametrize('dtype', [BF, HF])
def test_reference_maximum_covers_a_whole_tile(dtype):
    """128 keys are one step of the 256-row tile, whose P is rounded against the row's true maximum.  Two steps of 64 keys
    must come as close to 64 bits as that computation, rounding for rounding, does (0.5 % for the order of sums)."""
    from aotriton_amd.autograd import attention
    B, H, S, D = 40, 16, 128, 64
    g = torch.Generator(device='cuda').manual_seed(0)
    q, k, v = (torch.randn(B, H, S, D, device='cuda', generator=g).to(dtype) for _ in range(3))
    o = attention(q, k, v, None, False, D ** -0.5, 0.0)[0]
    s = torch.matmul(q.double(), k.double().transpose(-1, -2).contiguous()) * D ** -0.5
    want = torch.matmul(torch.softmax(s, -1), v.double())
    p = torch.exp(s - s.amax(-1, keepdim=True)).float()
    same = (torch.matmul(p.to(dtype).float(), v.float()) / p.sum(-1, keepdim=True)).to(dtype)
    off = lambda x: ((x.double() - want).norm() / want.norm()).item()
    assert off(o) <= 1.005 * off(same)
