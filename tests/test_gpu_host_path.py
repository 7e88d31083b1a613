"""The native host path (csrc/torch/host.cpp) against the views it stands in for."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = 'cuda'


@pytest.mark.parametrize('count', [0, 1, 239, 240, 241, 481, 1030])
def test_words_reach_the_device(count):
    """fa_write_words carries 240 words per launch: counts around whole launches; the words past the end
    of the range stay as they were."""
    from aotriton_amd._lib import lib
    words = [(0x9E3779B9 * (i + 1)) & 0xFFFFFFFF for i in range(count)]
    dst = torch.full([count + 4], -7, device=DEV, dtype=torch.int32)
    err = lib.fa_write_words(dst.data_ptr(), (ctypes.c_uint32 * max(count, 1))(*words), count,
                             torch.cuda.current_stream().cuda_stream or None)
    assert err == 0
    got = dst.tolist()
    assert [x & 0xFFFFFFFF for x in got[:count]] == words and got[count:] == [-7] * 4


@pytest.mark.parametrize('dropout_p', [0.0, 0.3])
def test_native_operators_equal_the_views(dropout_p):
    """flash.attn_fwd / attn_bwd on plain tensors go through the native path, the params structs of the
    pyaotriton-shaped module through ctypes: same kernels, same bits."""
    from aotriton_amd import flash
    from _util import make_inputs
    ok = flash.hipError_t.hipSuccess
    B, Hq, Hk, Sq, Sk, D, sm, causal = 2, 4, 2, 77, 131, 64, 0.125, (50, 3)
    q, k, v, b, do = make_inputs(B, Hq, Hk, Sq, Sk, D, torch.bfloat16, DEV, seed=3, bias=True, bshd=True)
    u64 = lambda x: torch.tensor([x], device=DEV, dtype=torch.int64).view(torch.uint64)
    got = []
    for native in (True, False):
        o, L = torch.empty_like(q), torch.empty(B * Hq, Sq, device=DEV)
        dq, dk, dv, db = (torch.empty_like(t) for t in (q, k, v, b))
        sd, o1, so, oo = u64(5), u64(9), u64(0), u64(0)
        atomic = torch.zeros([1], device=DEV, dtype=torch.int32)
        fwd = (q, k, v, b, sm, L, o, dropout_p, sd, o1, 3, so, oo, None, causal, atomic)
        bwd = (q, k, v, b, sm, o, do, dq, dk, dv, db, None, L, flash.lazy_delta(L), dropout_p, so, oo, 0, causal)
        if native:
            assert flash.attn_fwd(*fwd) == ok and flash.attn_bwd(*bwd) == ok
        else:
            p = flash.fa_forward_op_params()
            flash._fill_fwd(p, *fwd)
            assert flash.fa_forward_op(p, p.kVersion, flash._stream(), None) == ok
            p = flash.fa_backward_op_params()
            flash._fill_bwd(p, *bwd)
            assert flash.fa_backward_op(p, p.kVersion, flash._stream(), None) == ok
        torch.cuda.synchronize()
        got.append((o, L, dq, dk, dv, db, so.view(torch.int64), oo.view(torch.int64)))
    for x, y in zip(*got):
        assert torch.equal(x, y)


def test_a_flag_without_a_truth_value_is_reported():
    """the error of the conversion, not a result returned with an error set"""
    import numpy as np
    from aotriton_amd.torch_ops import scaled_dot_product_attention as sdpa
    q = torch.zeros(1, 2, 16, 64, device=DEV, dtype=torch.bfloat16)
    with pytest.raises(ValueError, match='ambiguous'):
        sdpa(q, q, q, enable_gqa=np.ones(2))
