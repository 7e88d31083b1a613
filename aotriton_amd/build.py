"""Builds libaotriton_amd.so (hipcc for gfx950, cross-compiles without a GPU) and _torch_host.so (the
native host path between PyTorch and the library, host code only) in-tree.

Usage: python -m aotriton_amd.build [-j N] [--force]
"""
import argparse
import concurrent.futures
import glob
import os
import re
import shutil
import subprocess
import sys
import tempfile

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, 'csrc')
ROOT = os.path.dirname(HERE)
OBJ = os.path.join(CSRC, 'obj')
LIB = os.path.join(HERE, 'libaotriton_amd.so')
HOST_SRC = os.path.join(CSRC, 'torch', 'host.cpp')
HOST_LIB = os.path.join(HERE, '_torch_host.so')
HOST_STAMP = os.path.join(OBJ, '_torch_host.torch')      # the torch version it was built for
HIPCC = os.environ.get('HIPCC', '/opt/rocm/bin/hipcc')

COMMON = [
    '--offload-arch=gfx950', '-O3', '-std=c++17', '-fPIC', '-fvisibility=hidden',
    '-I', os.path.join(ROOT, 'include'), '-I', CSRC,
    # packed fp32 VALU ops are kept off on this target
    '-Xclang', '-target-feature', '-Xclang', '-packed-fp32-ops',
    '-Wno-unused-command-line-argument',
]


# Per-file additions.  The dQ kernels post-process MFMA results with the vector ALU; letting
# the register allocator keep those results in VGPRs saves the AGPR read per element (kernels held to
# 256 registers, two waves per SIMD, have their results there anyway).
EXTRA = {
    # the ILP-first scheduling strategy: dK/dV kernel of the headline shape -1..2 % (same-box A/B,
    # no spills either way); level on the forward and the dQ-from-dS kernel, which keep the default
    'fa_bwd_dkdv_d128.hip': ['-mllvm', '-amdgpu-sched-strategy=max-ilp'],
    'fa_bwd_dkdv_parts_d128.hip': ['-mllvm', '-amdgpu-sched-strategy=max-ilp'],
    'fa_bwd_dq_bias_d64.hip': ['-mllvm', '-amdgpu-mfma-vgpr-form'],
    # (scores in vector registers; the accumulators are asm operands and stay in accumulation registers.  The loads into LDS
    # written as asm name m0 among what they change, and the compiler notes at each that it reserves that register.)
    'fa_fwd_wide_d128.hip': ['-mllvm', '-amdgpu-mfma-vgpr-form', '-Wno-inline-asm'],
    'fa_bwd_wide_d128.hip': ['-mllvm', '-amdgpu-mfma-vgpr-form', '-Wno-inline-asm'],
    'fa_bwd_pair_d256.hip': ['-Wno-inline-asm'],
    'fa_bwd_dqs.hip': ['-Wno-inline-asm'],
    'fa_fwd_d256.hip': ['-Wno-inline-asm'],
    'fa_bwd_dq_d128.hip': ['-mllvm', '-amdgpu-mfma-vgpr-form'],
}

# The per-head-dim kernel files are compiled a second time with FA_PADDED = the head dim: the copies that
# serve head dims rounded up to the compiled one.
PADDED_RE = re.compile(r'fa_(fwd|fwd_rows|fwd_wide|bwd_dkdv|bwd_dkdv_parts|bwd_dq|bwd_dq_bias|bwd_wide|bwd_pair|bwd_fused)_d(\d+)\.hip$')
# ... and these a third time with 96 columns, for head dims above 64 and up to 96
COLS96_RE = re.compile(r'fa_(fwd|fwd_wide|bwd_dkdv|bwd_dq|bwd_wide)_d128\.hip$')


def sources():
    """(source file, extra defines, object name) per compilation."""
    out = []
    for f in sorted(os.listdir(CSRC)):
        if not (f.endswith('.hip') or f.endswith('.cpp')):
            continue
        out.append((f, [], f + '.o'))
        if m := PADDED_RE.match(f):
            out.append((f, ['-DFA_PADDED=' + m.group(2)], f + '.padded.o'))
        if COLS96_RE.match(f):
            out.append((f, ['-DFA_PADDED=96'], f + '.cols96.o'))
    return out


def _inputs(path, obj):
    """The files a compilation read, from the dependency file next to its object; None without one."""
    try:
        text = open(obj + '.d').read()
    except OSError:
        return None
    names = text.replace('\\\n', ' ').split(':', 1)[-1].split()
    return [path] + [n for n in names if not n.startswith('/opt/')]


def _compile(unit, force):
    src, defines, objname = unit
    obj = os.path.join(OBJ, objname)
    path = os.path.join(CSRC, src)
    inputs = _inputs(path, obj)
    if (not force and inputs and os.path.exists(obj) and all(os.path.exists(p) for p in inputs) and
            os.path.getmtime(obj) >= max(os.path.getmtime(p) for p in inputs)):
        return obj, '', 0
    # the compiler's listing of the kernels (on its way to the object) is looked at before the object is taken
    with tempfile.TemporaryDirectory(prefix='fa_build_') as tmp:
        made = os.path.join(tmp, objname)
        cmd = [HIPCC] + COMMON + EXTRA.get(src, []) + defines + ['-save-temps=obj', '-MD', '-MF', obj + '.d', '-x', 'hip', '-c',
                                                                 path, '-o', made]
        r = subprocess.run(cmd, capture_output=True, text=True)
        # the host pass does not know the packed-fp32 feature name; that note is noise
        err = '\n'.join(l for l in r.stderr.splitlines() if 'packed-fp32-ops' not in l)
        if r.returncode == 0:
            for listing in glob.glob(os.path.join(tmp, '*gfx950.s')):
                lost = masked_spills(open(listing).read())
                if lost:
                    return obj, err + f'\n{objname}: values moved while lanes are off: {lost}', 1
            shutil.move(made, obj)
    return obj, err, r.returncode


def _host_is_current(torch_version):
    """Whether the extension is there, newer than what it is built from, and built for this torch (its C++ ABI
    is another with every version)."""
    try:
        built_for = open(HOST_STAMP).read()
        newest = max(os.path.getmtime(p) for p in [HOST_SRC, os.path.join(ROOT, 'include', 'aotriton_amd', 'flash.h')])
        return built_for == torch_version and os.path.getmtime(HOST_LIB) >= newest
    except OSError:
        return False


def build_host(force=False):
    """The Python extension over torch's C++ API.  It links against the library next to it."""
    import sysconfig
    import torch
    if not force and _host_is_current(str(torch.__version__)):
        return HOST_LIB
    from torch.utils import cpp_extension
    includes = cpp_extension.include_paths('cuda') + [sysconfig.get_paths()['include'], os.path.join(ROOT, 'include')]
    torch_lib = os.path.join(os.path.dirname(torch.__file__), 'lib')
    cmd = ['g++', '-O2', '-std=c++17', '-fPIC', '-shared', '-fvisibility=hidden', '-D__HIP_PLATFORM_AMD__=1', '-DUSE_ROCM=1',
           f'-D_GLIBCXX_USE_CXX11_ABI={int(torch.compiled_with_cxx11_abi())}', f'-DFA_TORCH_VERSION="{torch.__version__}"', '-Wno-deprecated-declarations',
           *[x for i in includes for x in ('-isystem', i)], HOST_SRC, '-o', HOST_LIB,
           '-L' + HERE, '-laotriton_amd', '-Wl,-rpath,$ORIGIN', '-L' + torch_lib, '-ltorch_python', '-ltorch', '-ltorch_cpu',
           '-ltorch_hip', '-lc10_hip', '-lc10']
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        sys.stderr.write(r.stderr)
        raise RuntimeError('g++ failed on ' + HOST_SRC)
    os.makedirs(OBJ, exist_ok=True)
    with open(HOST_STAMP, 'w') as f:
        f.write(torch.__version__)
    return HOST_LIB


def build(jobs=8, force=False, verbose=True):
    os.makedirs(OBJ, exist_ok=True)
    srcs = sources()
    objs = []
    failed = False
    with concurrent.futures.ThreadPoolExecutor(max_workers=jobs) as ex:
        for obj, err, rc in ex.map(lambda s: _compile(s, force), srcs):
            objs.append(obj)
            if err.strip() and (rc != 0 or verbose):
                sys.stderr.write(err + '\n')
            failed |= rc != 0
    if failed:
        raise RuntimeError('hipcc failed')
    cmd = [HIPCC, '--offload-arch=gfx950', '-shared', '-fPIC', '-o', LIB] + objs
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        sys.stderr.write(r.stderr)
        raise RuntimeError('link failed')
    build_host(force)
    return LIB


_WATERFALL = re.compile(r'v_readfirstlane_b32[^\n]*\n(?:[^\n]*\n){0,24}?[^\n]*s_and_saveexec_b64[^\n]*\n'
                        r'(?:[^\n]*\n){0,24}?[^\n]*buffer_(?:load|store)[^\n]*\n(?:[^\n]*\n){0,4}?'
                        r'[^\n]*s_xor_b64 exec, exec[^\n]*\n[^\n]*s_cbranch_execnz')


def masked_spills(text):
    """Vector instructions between the label where the lanes of a branch meet again and the instruction that turns them on:
    values the register allocator moved or spilled there.  hipcc 7.2 does so when a scalar move or reload stands in front of that
    instruction (it takes the block's prologue to end there); the lanes that are off keep what the new place held before, and a
    pointer among such values faults.  Found in the dQ kernel for padded head dims above 128 with a window and a bias, whose lanes
    32-63 stored dQ through such a pointer.  Returns (kernel, instruction) pairs."""
    joins = set(re.findall(r'^\s*s_cbranch_execz (\.LBB\w+)', text, re.M))
    found, head, before, kernel = [], None, '', ''
    for line in text.splitlines():
        block = re.match(r'(\.LBB\w+):|; (%bb\.\d+):', line.strip())
        if block:
            # (a block without a label and behind no jump is a meeting place whose jump was removed)
            falls_in = block.group(1) is None and not before.startswith(('s_cbranch', 's_branch', 's_endpgm', 's_setpc'))
            head = [] if block.group(1) in joins or falls_in else None
            continue
        if re.match(r'\w+:', line):
            kernel = line.split(':')[0]
        line = line.split(';')[0].strip()
        if not line or line.startswith('.') or line.endswith(':'):
            continue
        if head is not None:
            op = line.split()[0]
            if op.startswith(('s_cbranch', 's_branch', 's_endpgm')) or re.match(r's_\w+ exec,|s_\w+saveexec', line):
                if line.startswith('s_or_b64 exec, exec,'):
                    found += [(kernel, x) for x in head]
                head = None
            elif (op.startswith(('v_', 'scratch_', 'global_', 'buffer_', 'flat_', 'ds_')) and
                  not op.startswith(('v_readlane', 'v_writelane', 'v_readfirstlane', 'v_cmp'))):
                head.append(line)
        before = line
    return found


def asm_mfma_hazards(text):
    """MFMAs written as asm whose operands a vector instruction writes less than two instructions before: the compiler keeps
    that distance for its own MFMAs and does not look into asm.  Returns the lines."""
    def registers(operand):
        m = re.match(r'v\[(\d+):(\d+)\]$', operand) or re.match(r'v(\d+)()$', operand)
        return set(range(int(m.group(1)), int(m.group(2) or m.group(1)) + 1)) if m else set()
    found, before, in_asm = [], [], False
    for line in text.splitlines():
        if '#ASM' in line:
            in_asm = 'START' in line
        line = line.split(';')[0].strip()
        if not line or line.startswith('.') or line.endswith(':'):
            continue
        op, _, rest = line.partition(' ')
        args = [a.strip() for a in rest.split(',')]
        if in_asm and op.startswith('v_mfma'):
            sources, distance = registers(args[1]) | registers(args[2]), 0
            for written, states in reversed(before):
                if distance < 2 and written & sources:
                    found.append(line)
                distance += states
        vector = op.startswith('v_') and not op.startswith('v_mfma')
        before = (before + [(registers(args[0]) if vector else set(), int(args[0], 0) + 1 if op == 's_nop' else 1)])[-4:]
    return found


def asm_accumulator_hazards(text):
    """Instructions that read or write an accumulation register less than 20 wait states after an asm MFMA wrote it (16 passes and
    what the register file takes), on any path, except the next MFMA onto the same accumulator: the compiler keeps that
    distance behind its own MFMAs and does not look into asm.  Returns the lines.  (An MFMA counts as one state.)"""
    def accumulators(operand):
        m = re.match(r'a\[(\d+):(\d+)\]$', operand) or re.match(r'a(\d+)()$', operand)
        return frozenset(range(int(m.group(1)), int(m.group(2) or m.group(1)) + 1)) if m else frozenset()

    # blocks: [instructions (line, states, accumulators per operand, asm MFMA?), blocks that follow by label, falls through?]
    blocks, at, in_asm = [[[], [], True]], {}, False
    for line in text.splitlines():
        if '#ASM' in line:
            in_asm = 'START' in line
        line = line.split(';')[0].strip()
        if line.endswith(':') and (line.startswith('.LBB') or not line.startswith('.')):
            blocks.append([[], [], True])
            at[line[:-1]] = len(blocks) - 1
            blocks[-2][2] &= line.startswith('.')      # (not into the next kernel)
        if not line or line.startswith('.') or line.endswith(':'):
            continue
        op, _, rest = line.partition(' ')
        args = [a.split()[0] for a in rest.split(',')] if rest else []
        blocks[-1][0].append((line, int(args[0], 0) + 1 if op == 's_nop' else 1, [accumulators(a) for a in args],
                              in_asm and op.startswith('v_mfma')))
        if op.startswith(('s_cbranch', 's_branch', 's_endpgm', 's_setpc')):
            blocks[-1][1:] = [[args[0]] if 'branch' in op else [], op.startswith('s_cbranch')]
            blocks.append([[], [], True])

    # wait states since the last write of each accumulator, the fewest over all paths into a block
    found, entry, todo = {}, [{} for _ in blocks], set(range(len(blocks)))
    while todo:
        i = todo.pop()
        instructions, labels, falls = blocks[i]
        ages = dict(entry[i])
        for n, (line, states, used, asm_mfma) in enumerate(instructions):
            onto = used[0] if line.startswith('v_mfma') and used[3] in (used[0], frozenset()) else None
            if any(u & group and not u == onto == group for u in used for group in ages):
                found[i, n] = line
            ages = {group: age + states for group, age in ages.items() if age + states < 20}
            if asm_mfma and used[0]:
                ages[used[0]] = 0
        for j in [at[x] for x in labels if x in at] + ([i + 1] if falls and i + 1 < len(blocks) else []):
            merged = {g: min(ages.get(g, 20), entry[j].get(g, 20)) for g in {*ages, *entry[j]}}
            if merged != entry[j]:
                entry[j] = merged
                todo.add(j)
    return list(found.values())


def asm_memory_hazards(text):
    """Memory instructions that read a scalar register less than five wait states after a vector instruction wrote it: the
    compiler keeps that distance for its own and does not look into asm.  Returns the lines.  (Followed from line to line, so
    that what stands in front of a jump counts for the label behind it only.)"""
    def scalars(operand):
        m = re.match(r's\[(\d+):(\d+)\]$', operand) or re.match(r's(\d+)()$', operand)
        return range(int(m.group(1)), int(m.group(2) or m.group(1)) + 1) if m else ()
    found, written, now = [], {}, 0
    for line in text.splitlines():
        line = line.split(';')[0].strip()
        if not line or line.startswith('.') or line.endswith(':'):
            continue
        op, _, rest = line.partition(' ')
        args = [a.split()[0] for a in rest.split(',')] if rest else []
        if op.startswith(('buffer_', 'global_', 'flat_', 'scratch_')):
            if any(now - written.get(r, -5) < 5 for a in args for r in scalars(a)):
                found.append(line)
        now += int(args[0], 0) + 1 if op == 's_nop' else 1
        for a in args[:2] if op.startswith('v_') else args[:1] if op.startswith('s_') and not op.startswith('s_cmp') else ():
            for r in scalars(a):
                # (of the vector instructions that write a scalar register some have it in the second place)
                if op.startswith(('v_readlane', 'v_readfirstlane', 'v_cmp')) and a is args[0] or '_co_u32' in op or op.startswith(('v_mad_u64', 'v_mad_i64', 'v_div_scale')):
                    written[r] = now
                elif op.startswith('s_'):
                    written.pop(r, None)
    return found


def scan(jobs=8):
    """Compiles every kernel file to assembly and reports per-descriptor loops around buffer
    accesses ("waterfall" loops: readfirstlane, compare, masked issue, repeat while lanes are left).
    The compiler emits them when it takes a buffer descriptor for divergent, e.g. one built from
    threadIdx.x >> 6.  They cost time, and hipcc 7.2 has placed a register spill in the block such
    a loop exits to, before exec is restored: the store runs with no lane enabled and the reload
    later returns whatever the slot held.  The kernels here are written so that none is emitted;
    returns the list of (file, loops, functions left out of line, asm_mfma_hazards, asm_accumulator_hazards, asm_memory_hazards,
    masked_spills) that have some of any."""
    tmpdir = tempfile.TemporaryDirectory(prefix='fa_scan_')
    tmp = tmpdir.name

    def one(unit):
        src, defines, objname = unit
        if not src.endswith('.hip'):
            return src, 0, 0, [], [], [], []
        out = os.path.join(tmp, objname + '.s')
        cmd = [HIPCC] + COMMON + EXTRA.get(src, []) + defines + ['-x', 'hip', '--cuda-device-only', '-S',
                                                                 os.path.join(CSRC, src), '-o', out]
        r = subprocess.run(cmd, capture_output=True, text=True)
        if r.returncode != 0:
            raise RuntimeError('hipcc failed on ' + src)
        text = open(out).read()
        # a device function left out of line (a lambda the inliner gave up on) keeps its captures in
        # memory and reads them back with flat loads; every kernel here is meant to be one function
        outlined = len(re.findall(r'^\s*\.type\s+\S+,@function', text, re.M)) - text.count('.amdhsa_kernel ')
        return (objname, len(_WATERFALL.findall(text)), outlined, asm_mfma_hazards(text), asm_accumulator_hazards(text),
                asm_memory_hazards(text), masked_spills(text))

    with tmpdir, concurrent.futures.ThreadPoolExecutor(max_workers=jobs) as ex:
        return [r for r in ex.map(one, sources()) if any(r[1:])]


if __name__ == '__main__':
    ap = argparse.ArgumentParser()
    ap.add_argument('-j', type=int, default=8)
    ap.add_argument('--force', action='store_true')
    ap.add_argument('--scan', action='store_true', help='compile to assembly and look for per-descriptor loops')
    a = ap.parse_args()
    if a.scan:
        found = scan(a.j)
        print('per-descriptor loops / functions left out of line / asm MFMAs and memory accesses too close behind their operands or in front of what follows / values moved while lanes are off:', found if found else 'none')
        sys.exit(1 if found else 0)
    print(build(a.j, a.force))
