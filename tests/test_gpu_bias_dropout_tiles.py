"""Forward with a bias and dropout at head dims up to 128 in tiles of 128 rows, two workgroups per CU: ragged tiles on both sides, the fewest keys,
windows, rows at any alignment, against the oracle; and the tiles that calls get."""
import pytest
import torch

from test_gpu_attention import _run_case
from test_launch_queries import fwd

BF, HF = torch.bfloat16, torch.float16
CASES = [
    # B, Hq, Hk, Sq, Sk, D, dtype, causal
    (1, 2, 2, 513, 1, 64, BF, False),
    (1, 2, 1, 520, 7, 128, HF, False),            # fewer keys than a piece of a row
    (1, 2, 2, 514, 65, 64, HF, False),            # one key in the second tile
    (1, 4, 2, 641, 33, 128, BF, False),
    (2, 2, 2, 640, 640, 64, BF, True),            # whole tiles throughout
    (2, 2, 2, 640, 640, 128, HF, True),
    (1, 4, 2, 700, 531, 40, HF, (200, 40)),
    (1, 4, 4, 700, 531, 80, BF, (90, -30)),       # rows that see nothing
    (1, 2, 2, 577, 904, 96, HF, (100, 300)),
    (1, 2, 1, 800, 797, 128, BF, (300, 0)),
]


def _id(c):
    return '-'.join(str(x).replace('torch.', '') for x in c)


def test_cases_are_of_these_tiles():
    for c in CASES:
        x = fwd(*c[:6], c[7], 0.3, True)
        assert (x.block_m, x.block_n, x.num_waves) == (128, 64 if c[5] <= 64 else 32, 4), _id(c)
    for other in [(1, 2, 2, 512, 600, 64, False, 0.3, True), (1, 2, 2, 512, 600, 128, True, 0.3, True)]:
        assert fwd(*other).block_m == 256


@pytest.mark.gpu
@pytest.mark.parametrize('case', CASES, ids=_id)
def test_bias_and_dropout_meet_the_oracle(case):
    _run_case(*case, dropout_p=0.3, bias=True, seed=31)


@pytest.mark.gpu
@pytest.mark.parametrize('D,dt,causal', [(64, BF, (150, 20)), (64, HF, True), (128, BF, False), (96, HF, (77, 0))])
def test_rows_lie_anywhere(D, dt, causal):
    """Aligned rows, rows one element on and rows of an odd length: the same bits."""
    from aotriton_amd import flash
    B, H, Sq, Sk = 2, 2, 530, 421
    g = torch.Generator(device='cuda').manual_seed(7)
    rn = lambda *s: torch.randn(*s, device='cuda', generator=g).to(dt)
    q, k, v = rn(B, H, Sq, D), rn(B, H, Sk, D), rn(B, H, Sk, D)
    room = torch.full((B * H * Sq * Sk + 1,), float('nan'), device='cuda', dtype=dt)
    odd = room[1:].view(B, H, Sq, Sk).copy_(rn(B, H, Sq, Sk))
    wide = torch.full((B, H, Sq, 424), float('nan'), device='cuda', dtype=dt)
    wide[..., :Sk] = odd
    seed, off = (torch.tensor([x], device='cuda', dtype=torch.uint64) for x in (3, 4))
    null, got = torch.empty([0], device='cuda', dtype=torch.uint64), []
    for b in (odd, wide[..., :Sk], odd.contiguous().clone()):
        o, L = torch.empty_like(q), torch.empty(B * H, Sq, device='cuda')
        assert flash.attn_fwd(q, k, v, b, D ** -0.5, L, o, 0.2, seed, off, 0, null, null, None, causal, null) == flash.hipError_t.hipSuccess
        got.append((o, L))
    for o, L in got[1:]:
        assert torch.equal(o, got[0][0]) and torch.equal(L, got[0][1])


SHORT = [
    # rows for one tile of 256 at most
    (1, 8, 8, 64, 64, 64, BF, False),
    (5, 1, 1, 1, 129, 64, HF, False),             # one query
    (2, 4, 2, 31, 1, 128, BF, False),             # one key
    (3, 2, 2, 128, 96, 80, HF, True),
    (2, 3, 3, 129, 257, 128, HF, (40, 30)),       # one row in the second tile, one key in the last
    (1, 5, 5, 200, 333, 96, BF, (30, -10)),       # rows that see nothing
    (1, 3, 3, 256, 512, 40, HF, (128, 0)),
    (1, 6, 2, 256, 70, 64, BF, True),
]


def test_short_calls_are_of_these_tiles_too():
    for c in SHORT:
        x = fwd(*c[:6], c[7], 0.3, True)
        assert (x.block_m, x.block_n, x.num_waves) == (128, 64 if c[5] <= 64 else 32, 4), _id(c)


@pytest.mark.gpu
@pytest.mark.parametrize('case', SHORT, ids=_id)
def test_short_calls_meet_the_oracle(case):
    _run_case(*case, dropout_p=0.3, bias=True, seed=37)
