"""Forward with 64 rows per wave (long items at head dims 65-128) against the oracle: odd numbers of units and tiles, waves
whose windows start and end in different tiles, rows without a key, keys in parts, packed sequences, scores whose maximum
grows from unit to unit."""
import math

import numpy as np
import pytest
import torch

import test_gpu_fwd_tiles
from test_gpu_varlen_dropout import _run_varlen_case
from test_launch_queries import fwd, packed
from _util import make_inputs

BF, HF = torch.bfloat16, torch.float16
BR = (-2147483646, -2147483646)      # bottom right
CASES = [
    # B, Hq, Hk, Sq, Sk, D, dtype, causal, bias
    (4, 32, 32, 257, 1281, 128, BF, False, None),             # a second item of one row, a last tile of one key
    (4, 32, 8, 700, 1423, 128, HF, BR, None),
    (2, 32, 32, 1500, 1500, 128, BF, True, None),
    (4, 32, 32, 300, 1311, 96, HF, False, None),
    (4, 32, 32, 511, 1400, 72, BF, BR, None),
    (4, 32, 32, 300, 1300, 112, BF, (900, 700), None),
    (4, 32, 32, 400, 1300, 128, BF, (20, 1000), None),        # the last rows see no key
    (2, 32, 32, 600, 2400, 128, HF, (-700, 1500), None),      # the first tiles are seen by no row, waves start in different ones
]
SPLIT = [
    (1, 32, 32, 512, 6000, 128, BF, BR, None),
    (1, 24, 8, 600, 5555, 96, HF, False, None),
]


def _id(c):
    return '-'.join(str(x).replace('torch.', '') for x in c)


def test_cases_are_of_this_kernel():
    for case in CASES + SPLIT:
        c = fwd(*case[:6], case[7])
        assert (c.block_m, c.num_waves, c.flags & 192) == (256, 4, 64 if case in SPLIT else 0), _id(case)
    for other in [(16, 16, 16, 2048, 2048, 128, True), (4, 16, 16, 2048, 2048, 128, (256, 0)), (2, 32, 32, 1500, 1500, 64, True),
                  (2, 32, 32, 1500, 1500, 128, True, 0.1), (2, 32, 32, 1500, 1500, 128, True, 0.0, True)]:
        assert (fwd(*other).block_m, fwd(*other).num_waves) != (256, 4), other


@pytest.mark.gpu
@pytest.mark.parametrize('case', CASES + SPLIT, ids=_id)
def test_wide_forward_meets_the_oracle(case):
    test_gpu_fwd_tiles.test_forward_tiles_meet_the_oracle(case)


@pytest.mark.gpu
@pytest.mark.parametrize('dtype, top', [(BF, 3.0), (HF, 8.0), (BF, 60.0)])
def test_maximum_grows_from_unit_to_unit(dtype, top):
    """keys that grow along the sequence: every few units the speculative step fails and the full step moves the reference
    (top 60: scores beyond 1000, where the difference is formed first).  Against 64 bits: P and O are rounded to the type."""
    from aotriton_amd.autograd import attention
    q, k, v, _, _ = make_inputs(4, 32, 32, 300, 1300, 128, dtype, 'cuda', seed=2)
    k = k * torch.linspace(0.2, top, 1300, device='cuda').to(dtype).view(1, 1, -1, 1)
    o = attention(q, k, v, None, False, 1 / math.sqrt(128), 0.0)[0]
    torch.cuda.synchronize()
    x = [t[1, 5:9].double() for t in (q, k, v)]
    p = torch.softmax(x[0] @ x[1].transpose(1, 2).contiguous() / math.sqrt(128), -1)
    want = p @ x[2]
    eps = 2 ** -9 if dtype == BF else 2 ** -12
    # |error| <= eps (sum p |v| + |O|), twice that for the roundings of the operands' products and of the exponentials
    bound = 2 * eps * (p @ x[2].abs() + want.abs()) + 1e-3 * eps
    assert ((o[1, 5:9].double() - want).abs() <= bound).all()


@pytest.mark.gpu
@pytest.mark.parametrize('D, causal', [(128, True), (80, False), (128, (1200, 40))])
def test_wide_forward_of_packed_sequences(D, causal):
    lens = np.array([1411, 900, 0, 1800, 1290, 257, 2048, 1024])
    _run_varlen_case(lens, lens, 16, 8, D, BF, causal, 0, seed=8)


# lengths whose average brings the rule to these kernels: an empty sequence, ones that end with a row or a key in a tile of their own
PACKED = [np.array([1411, 900, 0, 1800, 1290, 257, 2048, 1024]), np.array([3001, 1, 2304, 0, 1345])]
PACKED_CASES = [(i, D, c, Hq, Hk) for D, c in [(128, True), (80, False), (128, (1200, 40)), (96, BR)] for i, Hq, Hk in [(0, 8, 4), (1, 8, 8)]]


def test_packed_cases_are_of_this_kernel():
    for i, D, causal, Hq, Hk in PACKED_CASES:
        c = packed(None, PACKED[i], PACKED[i][::-1] if causal == BR else PACKED[i], Hq, Hk, D, causal)
        assert (c.block_m, c.num_waves, c.flags & 192) == (256, 4, 0), (i, D, causal)


@pytest.mark.gpu
@pytest.mark.parametrize('i, D, causal, Hq, Hk', PACKED_CASES)
def test_packed_sequences_on_this_kernel_meet_the_oracle(i, D, causal, Hq, Hk):
    lens = PACKED[i]
    _run_varlen_case(lens, lens[::-1].copy() if causal == BR else lens, Hq, Hk, D, BF if i else HF, causal, 0, seed=18)
