"""The checks of the compiler's listings (build.py) on listings with a known answer: wait states that the compiler does not see to
because one of the two instructions stands in asm, also on the loads into LDS (fa_wide.h) compiled behind the instructions that
precede them; values that the register allocator moves while lanes are off."""
import os
import subprocess

import pytest

from aotriton_amd import build

LOAD = 'buffer_load_dwordx4 v5, s[4:7], s39 offen lds'


@pytest.mark.parametrize('between, found', [
    (['v_readlane_b32 s39, v254, 2', 's_mov_b32 m0, s50', 's_nop 0'], 1),
    (['v_readfirstlane_b32 s7, v1', 's_mov_b32 m0, s50', 's_nop 2'], 1),
    (['v_cmp_gt_u32_e64 s[6:7], v0, v1', 's_mov_b32 m0, s50', 's_nop 0'], 1),
    (['v_readlane_b32 s39, v254, 2', 's_mov_b32 m0, s50', 's_nop 3'], 0),
    (['v_readlane_b32 s39, v254, 2', 's_mov_b32 s39, s3', 's_nop 0'], 0),      # written again by a scalar instruction
    (['v_readlane_b32 s8, v254, 2', 's_nop 0'], 0),                           # another register
    (['v_add_u32_e32 v5, s39, v5', 's_nop 0'], 0),                            # read, not written
])
def test_memory_hazards_of_a_listing(between, found):
    assert len(build.asm_memory_hazards('\n'.join(f'\t{x}' for x in between + [LOAD]))) == found


MFMA = [';;#ASMSTART', 'v_mfma_f32_32x32x16_bf16 a[0:15], v[2:5], v[6:9], a[0:15]', ';;#ASMEND']


@pytest.mark.parametrize('behind, found', [
    (['s_nop 15', 's_nop 2', 'v_accvgpr_read_b32 v1, a3'], 1),
    (['s_nop 15', 's_nop 3', 'v_accvgpr_read_b32 v1, a3'], 0),
    (['v_accvgpr_write_b32 a15, v1'], 1),
    (['v_accvgpr_write_b32 a16, v1', 'global_store_dword v[2:3], a40, off'], 0),      # other registers
    (['global_store_dword v[2:3], a4, off'], 1),
    (['v_mfma_f32_32x32x16_bf16 a[0:15], v[2:5], v[6:9], a[0:15]'], 0),               # onto the same accumulator
    (['v_mfma_f32_32x32x16_bf16 v[20:35], a[12:15], v[6:9], 0'], 1),                  # as an operand
    (['v_mfma_f32_32x32x16_bf16 a[8:23], v[2:5], v[6:9], a[8:23]'], 1),               # a part of it
    # out of a loop to where its results are read, with and without a wait there
    (['s_cbranch_scc1 .LBB0_2', 's_nop 15', 's_nop 15', '.LBB0_2:', 'v_accvgpr_read_b32 v1, a3'], 1),
    (['s_cbranch_scc1 .LBB0_2', 's_branch .LBB0_3', '.LBB0_2:', 's_nop 15', 's_nop 3', '.LBB0_3:', 'v_mov_b32 v1, v2'], 0),
    (['s_branch .LBB0_3', '.LBB0_2:', 'v_accvgpr_read_b32 v1, a3', 's_endpgm', '.LBB0_3:', 's_nop 15', 's_nop 3', 's_branch .LBB0_2'], 0),
])
def test_accumulator_hazards_of_a_listing(behind, found):
    assert len(build.asm_accumulator_hazards('\n'.join(f'\t{x}' for x in MFMA + behind))) == found


def test_loads_into_lds_wait_for_their_scalars(tmp_path):
    """descriptor and offset come out of vector registers right in front of the load"""
    (tmp_path / 'x.hip').write_text('''#include "fa_wide.h"
__global__ void k(const char* p, const int* n) {
  extern __shared__ char smem[];
  const int t = threadIdx.x, o = n[t];
  fa::load_to_lds(fa::wave_rsrc_words(p + o, o), t * 16, __builtin_amdgcn_readfirstlane(o + 1), fa::lds_offset(smem),
                  t * 16, __builtin_amdgcn_readfirstlane(o + 2), fa::lds_offset(smem) + 1024);
}
''')
    if not os.path.exists(build.HIPCC):
        pytest.skip('no hipcc')
    out = tmp_path / 'x.s'
    subprocess.run([build.HIPCC] + build.COMMON + ['-x', 'hip', '--cuda-device-only', '-S', str(tmp_path / 'x.hip'), '-o', str(out)],
                   check=True, capture_output=True)
    text = out.read_text()
    assert text.count('offen lds') == 2 and 'v_readfirstlane' in text
    assert build.asm_memory_hazards(text) == []


def listing(*between, meeting='.LBB6_108:'):
    return '\n'.join(['_ZN2fa6kernelEv:', '\ts_and_saveexec_b64 s[4:5], s[8:9]', '\ts_cbranch_execz .LBB6_108', '; %bb.107:',
                      '\tglobal_store_dword v[4:5], v2, off', meeting] + [f'\t{x}' for x in between] + ['\ts_or_b64 exec, exec, s[4:5]',
                                                                                                    '\tv_mov_b32_e32 v1, v3'])


@pytest.mark.parametrize('text, found', [
    (listing('v_accvgpr_write_b32 a205, v31', 'v_accvgpr_write_b32 a204, v30', 's_mov_b32 s93, s87'), 2),
    (listing('s_mov_b64 s[98:99], s[64:65]', 'scratch_store_dwordx2 off, v[250:251], off offset:72 ; 8-byte Folded Spill'), 1),
    (listing('v_mov_b32_e32 v7, v8', meeting='; %bb.108:'), 1),
    (listing('s_mov_b32 s93, s87', 'v_readlane_b32 s5, v254, 25', 'v_writelane_b32 v253, s97, 2', 's_waitcnt vmcnt(0)'), 0),      # scalars
    (listing(), 0),
    # the lanes' own work, with the meeting point's instruction at its end
    ('_ZN2fa6kernelEv:\n\ts_cbranch_execz .LBB2_50\n.LBB2_53:\n\tv_add_u32_e32 v2, v2, v252\n\ts_or_b64 exec, exec, s[16:17]', 0),
])
def test_values_moved_while_lanes_are_off(text, found):
    got = build.masked_spills(text)
    assert len(got) == found and all(k == '_ZN2fa6kernelEv' for k, _ in got)
