"""The range of a buffer descriptor over a tile's rows (fa_intervals.h: rows_extent), compiled for the host: it ends with the
tensor's last row and is empty where there is no row, also for views whose rows overlap (an unfold, an expand)."""
import ctypes
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), 'aotriton_amd', 'csrc')


@pytest.fixture(scope='module')
def rows_extent(tmp_path_factory):
    if shutil.which('g++') is None:
        pytest.skip('no host compiler')
    d = tmp_path_factory.mktemp('rows_extent')
    (d / 'x.cpp').write_text('#include "fa_intervals.h"\n'
                             'extern "C" int rows_extent(int rows, int row, int head) { return fa::rows_extent(rows, row, head); }\n')
    subprocess.run(['g++', '-O2', '-std=c++17', '-shared', '-fPIC', '-fwrapv', '-I', CSRC, str(d / 'x.cpp'), '-o', str(d / 'x.so')], check=True)
    return ctypes.CDLL(str(d / 'x.so')).rows_extent


@pytest.mark.parametrize('head', [144, 192, 256])
@pytest.mark.parametrize('row', [0, 16, 128, 256, 8192, 1 << 22])
def test_ends_with_the_last_row(rows_extent, row, head):
    for rows in range(-70, 65):
        assert rows_extent(rows, row, head) == ((rows - 1) * row + head if rows > 0 else 0), rows


@pytest.mark.parametrize('row', [0, 128, 256])
def test_requests_stay_inside_the_tensor(rows_extent, row):
    """a walk over 1300 rows in tiles of 32 and 64 and two requests behind the last tile, as the wide kernels make them"""
    n, head = 1300, 256
    end = (n - 1) * row + head
    for tile in (32, 64):
        for t in range((n + tile - 1) // tile + 2):
            size = rows_extent(min(n - t * tile, tile), row, head)
            assert size >= 0 and (size == 0 or t * tile * row + size <= end), t


def test_stride_of_a_single_row_does_not_matter(rows_extent):
    for row in (-(1 << 31), -4096, 1 << 30, (1 << 31) - 1):
        assert rows_extent(1, row, 256) == 256 and rows_extent(0, row, 256) == 0


def overlapping(B, H, S, D, row, dtype, seed):
    """(B, H, S, D) whose rows start every `row` elements, the last one at the end of the memory"""
    import torch
    n = (S - 1) * row + D
    flat = torch.randn(B, H, n, generator=torch.Generator().manual_seed(seed)).to(dtype).cuda()
    return flat.as_strided((B, H, S, D), (H * n, n, row, 1))


@pytest.mark.gpu
@pytest.mark.parametrize('causal', [False, (900, 700)])
@pytest.mark.parametrize('D, row', [(128, 64), (96, 8)])
def test_wide_kernels_read_overlapping_rows(D, row, causal):
    """Q, K and V as overlapping views, dO the same row for all tokens: the results of their contiguous copies, to the bit"""
    import torch
    from aotriton_amd.autograd import attention
    from test_launch_queries import bwd, fwd
    shape = (4, 32, 32, 300, 1300, D)
    B, H, _, Sq, Sk, _ = shape
    assert (fwd(*shape, causal).block_m, fwd(*shape, causal).num_waves) == (256, 4)
    assert bwd(1, *shape, causal).block_n == 256 and bwd(2, *shape, causal).block_m == 256
    q, k, v = (overlapping(B, H, S, D, row, torch.bfloat16, i) for i, S in enumerate((Sq, Sk, Sk)))
    do = overlapping(B, H, 1, D, 0, torch.bfloat16, 3).expand(B, H, Sq, D)
    got = []
    for copy in (False, True):
        x = [(t.contiguous() if copy else t).detach().requires_grad_() for t in (q, k, v)]
        assert copy or x[1].stride() == k.stride()
        o = attention(*x, None, causal, D ** -0.5, 0.0)[0]
        o.backward(do.contiguous() if copy else do)
        got.append([o] + [t.grad for t in x])
    torch.cuda.synchronize()
    for a, b in zip(*got):
        assert torch.isfinite(a).all() and torch.equal(a, b)
