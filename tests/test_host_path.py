"""What the native host path (csrc/torch/host.cpp) checks before anything reaches a device; meta tensors
stand in for GPU ones."""
import numpy as np
import pytest
import torch


def _meta(*shape):
    return torch.empty(*shape, dtype=torch.bfloat16, device='meta')


@pytest.mark.parametrize('lens_q, lens_k', [
    ([7, 8], [10, 14]),         # one query row short: it would stay unwritten
    ([8, 9], [10, 14]),         # one too many: past the end of the tensors
    ([8, 8], [10, 13]),
    ([8, 8], [10, 15]),
    ([20, -4], [10, 14]),       # the sums are right, the lengths are not
    ([8, 8], [-1, 25]),
    ([], []),
    ([2 ** 32 + 16], [24]),     # equal to the tokens in 32 bits
])
def test_packed_lengths_must_add_up(lens_q, lens_k):
    from aotriton_amd.autograd import attention_varlen
    q, k = _meta(1, 4, 16, 64), _meta(1, 2, 24, 64)
    with pytest.raises(ValueError):
        attention_varlen(q, k, k, lens_q, lens_k, False, 0.125, 0.0)


@pytest.mark.parametrize('lens', [[16.0], np.array([16.0, 0.0]), [[10, 6]], np.array([[4], [12]], np.int32),
                                  torch.tensor([16]), np.array([16], np.uint64), (9, 7)])
def test_packed_lengths_of_any_shape_and_number_type(lens):
    """they get past the reading of the lengths: what is refused is the key side"""
    from aotriton_amd.autograd import attention_varlen
    q, k = _meta(1, 4, 16, 64), _meta(1, 2, 24, 64)
    with pytest.raises(ValueError, match='key sequence lengths add up to 23'):
        attention_varlen(q, k, k, lens, [10, 13], False, 0.125, 0.0)
