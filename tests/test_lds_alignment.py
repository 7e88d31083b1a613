"""Kernels that pick LDS operands by an exclusive or with an absolute address declare their LDS so aligned that it leaves the bits of the
base alone.  It lies at address 0 today; a static array in front of it would move it."""
import os
import re

import pytest

from aotriton_amd import build

SWZ_BITS = 256      # fa_device.h: a swizzle moves chunks inside this many bytes


def _read(name):
    return re.sub(r'//[^\n]*', '', open(os.path.join(build.CSRC, name)).read())


@pytest.mark.parametrize('item, kernel', [('fa_fwd_pair.h', 'fa_fwd_impl.h'), ('fa_bwd_pair.h', 'fa_bwd_pair.h')])
def test_lds_of_kernels_that_swizzle_addresses(item, kernel):
    assert 'lds_offset(smem_raw)' in _read(item) and re.search(r'_at \^', _read(item))
    declared = re.findall(r'__shared__ __attribute__\(\(aligned\((.*)\)\)\) char smem_raw', _read(kernel))
    align = int(re.search(r'kSwzAlign = (\d+)', _read('fa_device.h')).group(1))
    assert len(declared) == 1 and align >= SWZ_BITS
    assert declared[0] == 'kPairs ? kSwzAlign : 16' or int(declared[0]) >= SWZ_BITS


def test_no_other_kernel_swizzles_addresses():
    found = {f for f in os.listdir(build.CSRC) if f.endswith(('.h', '.hip')) and re.search(r'_at \^', _read(f))}
    assert found == {'fa_fwd_pair.h', 'fa_bwd_pair.h'}
