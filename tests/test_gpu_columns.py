"""Head dims above 64 and up to 96 compute 96 of the 128 columns of their build.  Against the oracle at
the edges of that range, with unequal head dims on either side of it, options, and a ragged last tile."""
import pytest
import torch

from test_gpu_attention import _run_case

pytestmark = pytest.mark.gpu

BF, HF = torch.bfloat16, torch.float16
CASES = [
    # Hq, Hk, Sq, Sk, D, Dv, dtype, causal, dropout, bias
    (2, 2, 300, 270, 72, None, BF, False, 0.0, False),
    (4, 2, 257, 129, 96, None, HF, True, 0.0, False),
    (2, 1, 200, 333, 88, None, HF, (50, 20), 0.1, False),
    (2, 2, 131, 190, 80, None, BF, False, 0.0, True),
    (2, 2, 190, 131, 96, None, HF, True, 0.2, True),
    (2, 2, 150, 260, 96, 72, BF, True, 0.1, False),
    (2, 2, 150, 260, 96, 104, BF, False, 0.0, False),        # V needs the 128 columns
    (2, 2, 260, 150, 104, 96, HF, True, 0.1, False),         # Q and K do
    (2, 2, 150, 150, 40, 80, HF, False, 0.0, False),
]


@pytest.mark.parametrize('case', CASES, ids=lambda c: '-'.join(str(x).replace('torch.', '') for x in c))
def test_columns_meet_the_oracle(case, with_and_without_workspace):
    Hq, Hk, Sq, Sk, D, Dv, dtype, causal, p, bias = case
    _run_case(2, Hq, Hk, Sq, Sk, D, dtype, causal, dropout_p=p, bias=bias, Dv=Dv, seed=17)
