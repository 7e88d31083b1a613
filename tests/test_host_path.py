"""What the native host path (csrc/torch/host.cpp) checks before anything reaches a device; meta tensors
stand in for GPU ones."""
import os
import subprocess
import sys

import numpy as np
import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


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


@pytest.mark.parametrize('requires_grad', [False, True])
@pytest.mark.parametrize('entry, dual', [(e, d) for e in ('attention', 'attention_varlen', 'sdpa') for d in 'qkvb'
                                         if (e, d) != ('attention_varlen', 'b')])      # (that one takes no bias)
def test_forward_mode_is_refused(entry, dual, requires_grad):
    """a tangent must not be dropped, with or without a gradient to record"""
    import torch.autograd.forward_ad as fwad
    from aotriton_amd.autograd import attention, attention_varlen
    from aotriton_amd.sdpa import scaled_dot_product_attention
    t = {'q': _meta(1, 4, 16, 64), 'k': _meta(1, 4, 24, 64), 'v': _meta(1, 4, 24, 64), 'b': _meta(1, 4, 16, 24)}
    for x in t.values():
        x.requires_grad_(requires_grad)
    with fwad.dual_level():
        t[dual] = fwad.make_dual(t[dual], torch.empty_like(t[dual]))
        with pytest.raises(NotImplementedError, match='forward-mode'):
            if entry == 'attention':
                attention(t['q'], t['k'], t['v'], t['b'], False, 0.125, 0.0)
            elif entry == 'attention_varlen':
                attention_varlen(t['q'], t['k'], t['v'], [16], [24], False, 0.125, 0.0)
            else:
                scaled_dot_product_attention(t['q'], t['k'], t['v'], t['b'])


def test_forward_mode_of_the_ops_is_refused_with_a_gradient():
    import torch.autograd.forward_ad as fwad
    from aotriton_amd.torch_ops import flash_attention_backward, scaled_dot_product_attention
    q, k = _meta(1, 4, 16, 64).requires_grad_(), _meta(1, 4, 24, 64)
    s, lse = torch.empty(1, dtype=torch.uint64, device='meta'), torch.empty(4, 16, device='meta')
    with fwad.dual_level():
        d = fwad.make_dual(q, torch.empty_like(q))
        with pytest.raises(NotImplementedError, match='forward-mode'):
            scaled_dot_product_attention(d, k, k)
        with pytest.raises(NotImplementedError, match='forward-mode'):
            flash_attention_backward(q.detach(), d, k, k, None, q.detach(), lse, 0.0, 0, 0, 0, 0.1, s, s, False, -1)


def _in_a_new_interpreter(blocked, code):
    code = f"import sys\nsys.modules[{blocked!r}] = None\n{code}"
    return subprocess.run([sys.executable, '-c', code], cwd=ROOT, capture_output=True, text=True)


@pytest.mark.parametrize('blocked', ['torch', 'aotriton_amd._torch_host'])
def test_flash_imports_without_torch_or_the_extension(blocked):
    """the constants, the params and the views are of use without either"""
    r = _in_a_new_interpreter(blocked, 'from aotriton_amd import flash\nprint(flash.translate_causal((5, 7)), flash.get_name_suffix())')
    assert r.returncode == 0, r.stderr
    assert r.stdout.split() == ['(3,', '5,', '7)', '_amd_gfx950']


@pytest.mark.parametrize('use', ['aotriton_amd.autograd', 'aotriton_amd.torch_ops',
                                 'aotriton_amd.flash; aotriton_amd.flash.attn_fwd(*[None] * 14, False, None)'])
def test_a_missing_extension_is_reported_with_the_way_to_build_it(use):
    r = _in_a_new_interpreter('aotriton_amd._torch_host', f'import {use}')
    assert r.returncode != 0 and 'ImportError' in r.stderr and 'python -m aotriton_amd.build' in r.stderr


def test_the_extension_is_rebuilt_for_another_torch(tmp_path, monkeypatch):
    from aotriton_amd import build
    ran = []
    monkeypatch.setattr(build, 'OBJ', str(tmp_path))
    monkeypatch.setattr(build, 'HOST_LIB', str(tmp_path / 'ext.so'))
    monkeypatch.setattr(build, 'HOST_STAMP', str(tmp_path / 'ext.torch'), raising=False)
    monkeypatch.setattr(build.subprocess, 'run', lambda cmd, **kw: ran.append(cmd) or subprocess.CompletedProcess(cmd, 0))
    (tmp_path / 'ext.so').touch()      # newer than the sources, built for nobody knows which torch
    build.build_host()
    assert len(ran) == 1
    build.build_host()
    assert len(ran) == 1
    monkeypatch.setattr(torch, '__version__', '0.0.0')
    build.build_host()
    assert len(ran) == 2


def test_an_extension_built_for_another_torch_is_refused(monkeypatch):
    from aotriton_amd import _host
    _host.load()
    monkeypatch.setattr(torch, '__version__', '0.0.0')
    with pytest.raises(ImportError, match='python -m aotriton_amd.build'):
        _host.load()
