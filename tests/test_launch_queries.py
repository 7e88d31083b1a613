"""fa_query_*_config reports the tile and grid of the kernel variant that a call runs on.  Host only: the views
point nowhere and nothing is launched."""
import pytest

CAUSAL = (3, -2147483647, -2147483647)


def view(*sizes, name='kBFloat16'):
    from aotriton_amd.pyaotriton import DType, T1, T2, T4
    strides = [1]
    for n in reversed(sizes[1:]):
        strides.insert(0, strides[0] * n)
    return {1: T1, 2: T2, 4: T4}[len(sizes)](4096, list(sizes), strides, getattr(DType, name))


def fwd(B, Hq, Hk, Sq, Sk, D, causal=False, p=0.0, bias=False, num_cu=256):
    from aotriton_amd.pyaotriton.v3.flash import attn_fwd_params, query_fwd_config
    x = attn_fwd_params()
    x.Q, x.K, x.V, x.Out = view(B, Hq, Sq, D), view(B, Hk, Sk, D), view(B, Hk, Sk, D), view(B, Hq, Sq, D)
    _common(x, B, Hq, Sq, Sk, causal, p, bias)
    err, c = query_fwd_config(x, num_cu)
    assert int(err) == 0
    return c


def bwd(slot, B, Hq, Hk, Sq, Sk, D, causal=False, p=0.0, bias=False, db=False, at=0):
    """bias: whether there is one, or its strides (`at` bytes behind a 16-byte boundary); db: the gradient is laid out as it is"""
    from aotriton_amd.pyaotriton.v3.flash import attn_bwd_params, query_bwd_config
    from aotriton_amd.pyaotriton import DType, T4, lazy_tensor
    x = attn_bwd_params()
    x.Q = x.DQ = view(B, Hq, Sq, D)
    x.Out = x.DO = view(B, Hq, Sq, D)
    x.K = x.V = x.DK = x.DV = view(B, Hk, Sk, D)
    x.L = view(B * Hq, Sq, name='kFloat32')
    x.D = lazy_tensor.eager_delta(x.L)
    _common(x, B, Hq, Sq, Sk, causal, p, bias)
    if isinstance(bias, tuple):
        x.B = T4(4096 + at, [B, Hq, Sq, Sk], list(bias), DType.kBFloat16)
    if db:
        x.DB = x.B
    err, c = query_bwd_config(x, slot)
    assert int(err) == 0
    return c


def packed(slot, lens_q, lens_k, Hq, Hk, D, causal=False, longest=None, num_cu=256):
    """the configuration of packed sequences (compact), forward with slot None"""
    from aotriton_amd.pyaotriton.v3.flash import attn_bwd_params, attn_fwd_params, query_bwd_config, query_fwd_config
    from aotriton_amd.pyaotriton import lazy_tensor
    Sq, Sk = int(sum(lens_q)), int(sum(lens_k))
    x = attn_fwd_params() if slot is None else attn_bwd_params()
    x.Q = x.Out = view(1, Hq, Sq, D)
    x.K = x.V = view(1, Hk, Sk, D)
    if slot is not None:
        x.DQ, x.DO, x.DK, x.DV, x.L = x.Q, x.Q, x.K, x.K, view(Hq, Sq, name='kFloat32')
        x.D = lazy_tensor.eager_delta(x.L)
    _common(x, 1, Hq, Sq, Sk, causal, 0.0, False)
    x.cu_seqlens_q = x.cu_seqlens_k = view(len(lens_q) + 1, name='kInt32')
    x.varlen_type = 1
    x.Max_seqlen_q, x.Max_seqlen_k = longest or int(max(lens_q)), longest or int(max(lens_k))
    err, c = query_fwd_config(x, num_cu) if slot is None else query_bwd_config(x, slot)
    assert int(err) == 0
    return c


def _common(x, B, Hq, Sq, Sk, causal, p, bias):
    from aotriton_amd.pyaotriton import DType, T0
    x.Sm_scale = 0.125
    if bias:
        x.B = view(B, Hq, Sq, Sk)
    x.dropout_p = p
    if p:
        x.philox_seed_ptr = x.philox_offset1 = T0(4096, DType.kUInt64)
    if causal:
        x.causal_type, x.window_left, x.window_right = CAUSAL if causal is True else (3, *causal)


def test_forward_variants():
    full = fwd(4, 32, 32, 4096, 4096, 64)
    assert (full.block_m, full.num_waves, full.grid[0], full.flags & 192) == (256, 8, 256, 0)
    half = fwd(40, 16, 16, 128, 128, 64, p=0.1)                 # 128-row tiles, two workgroups per CU
    assert (half.block_m, half.block_n, half.num_waves, half.grid[0]) == (128, 64, 4, 512)
    assert half.lds_bytes < 80 * 1024
    chunk = fwd(1, 32, 32, 1024, 16384, 128, causal=(-2147483646, -2147483646))      # tiles with their keys in parts
    assert (chunk.block_m, chunk.grid[0], chunk.flags & 192) == (256, 256, 64)
    few = fwd(1, 4, 4, 256, 8192, 128, p=0.0)
    assert few.grid[0] > 8 * ((4 + 7) // 8) and few.flags & 64   # more workgroups than tiles
    decode = fwd(1, 32, 8, 1, 4000, 128)
    assert decode.flags & 192 == 192
    assert fwd(1, 32, 8, 1, 4000, 128, p=0.1).flags & 192 == 0   # dropout stays on the tile kernel


@pytest.mark.parametrize('slot, bias, p, stored, tile, lds, grid', [
    (1, False, 0.0, False, (64, 128), 72704, 512),
    (1, False, 0.1, True, (64, 128), 72704, 512),
    (1, True, 0.0, True, (64, 128), 72704, 2048),                # one workgroup per item with a bias; 64-query steps storing dS,
    (1, True, 0.0, False, (128, 128), 141312, 2048),             # 128 recomputing it
    (1, True, 0.1, True, (64, 128), 72704, 2048),
    (1, True, 0.1, False, (64, 128), 72704, 2048),
    (2, False, 0.0, False, (128, 64), 51200, 512),
    (2, True, 0.0, True, (128, 128), 100352, 2048),
    (3, False, 0.0, False, (128, 128), 137216, 256),
    (3, True, 0.1, False, (128, 128), 137216, 4096),
])
def test_backward_variants_at_head_dim_64(slot, bias, p, stored, tile, lds, grid):
    from aotriton_amd._lib import lib
    lib.fa_set_bwd_workspace_limit(-1 if stored else 0)
    try:
        c = bwd(slot, 8, 16, 16, 2048, 2048, 64, bias=bias, p=p)
    finally:
        lib.fa_set_bwd_workspace_limit(-1)
    assert ((c.block_m, c.block_n), c.lds_bytes, c.grid[0]) == (tile, lds, grid)


def test_backward_parts_are_counted():
    whole, cut = bwd(1, 1, 8, 8, 64, 200, 128), bwd(1, 1, 8, 2, 1500, 200, 128)
    assert whole.flags & 64 == 0 and whole.grid[0] == 8 * 4      # a pair of heads per XCD, two key tiles each
    assert cut.flags & 64 and cut.grid[0] > 8 * 4
    from aotriton_amd._lib import lib
    lib.fa_set_bwd_workspace_limit(0)
    try:
        uncut = bwd(1, 1, 8, 2, 1500, 200, 128)
        assert uncut.flags & 64 == 0 and uncut.grid[0] == 8 * 4
    finally:
        lib.fa_set_bwd_workspace_limit(-1)


@pytest.mark.parametrize('call, db, parts', [
    ((2, 8, 1024, 1024), False, 2), ((1, 8, 1024, 1024), False, 4), ((1, 8, 512, 512), False, 4), ((4, 16, 256, 256), False, 1),
    ((3, 2, 2247, 151), False, 10), ((1, 12, 2304, 128), False, 10),      # the finest cut within 2 % of the lowest estimate: 9 parts, not of another cut
    # dB of a small call: dS is not stored
    ((1, 2, 1024, 1024), True, 4), ((1, 8, 512, 512), True, 2), ((3, 2, 2247, 151), True, 9), ((1, 2, 1400, 1400), True, 4),
    ((1, 3, 900, 900), True, 4), ((1, 8, 256, 256), True, 1),
])
def test_parts_share_cus_only_where_ds_is_stored(call, db, parts):
    """head dim 64 with a bias: level estimates are a gain for the kernels with two workgroups per CU, and cost the others up to 16 %"""
    from aotriton_amd._lib import lib
    B, H, Sq, Sk = call
    cut = bwd(1, B, H, H, Sq, Sk, 64, bias=True, db=db).grid[0]
    lib.fa_set_bwd_workspace_limit(0)
    try:
        assert cut == parts * bwd(1, B, H, H, Sq, Sk, 64, bias=True, db=db).grid[0]
    finally:
        lib.fa_set_bwd_workspace_limit(-1)


def _name(case):
    return '-'.join(str(x).replace('torch.', '') for x in case)


# the cases of the GPU tests are cases of the kernels that those tests are about
def test_cases_of_the_packed_rows_kernel():
    from test_gpu_fwd_rows import BR, CASES
    for B, Hq, Hk, Sq, Sk, D, _, causal, bias in CASES:
        c = fwd(B, Hq, Hk, Sq, Sk, (D + 7) // 8 * 8, (-2147483646, -2147483646) if causal == BR else causal, 0.0, bias)
        assert c.flags & 128, (B, Hq, Hk, Sq, Sk, D, causal)


def test_cases_of_the_forward_tiles():
    from test_gpu_fwd_tiles import SPLIT, TILES
    seen = set()
    for case in TILES + SPLIT:
        B, Hq, Hk, Sq, Sk, D, _, causal, bias = case
        c = fwd(B, Hq, Hk, Sq, Sk, D, causal, 0.0, bias is not None)
        assert c.flags & 192 == (64 if case in SPLIT else 0), _name(case)
        seen.add((c.head_dim, bool(causal), bias is not None, case in SPLIT, c.block_m if c.head_dim < 256 else 256))
    for D in (64, 128):      # every variant without dropout, with whole and half tiles
        for windowed in (False, True):
            assert {(D, windowed, False, False, 256), (D, windowed, False, False, 128), (D, windowed, True, False, 256),
                    (D, windowed, False, True, 256)} <= seen
    assert {(256, False, False, False, 256), (256, True, False, False, 256)} <= seen


def test_cases_of_the_half_tiles():
    from test_gpu_half_tiles import CASES
    half = [c for c in CASES if fwd(*c[:6], *c[7:]).flags & 192 == 0 and fwd(*c[:6], *c[7:]).block_m == 128]
    assert len(half) == 7 and {(c[5] > 64, bool(c[7]), c[8] > 0) for c in half} >= {
        (False, False, False), (False, True, True), (False, False, True), (True, True, False), (True, False, True)}


def test_cases_of_the_backward_parts():
    from test_gpu_bwd_parts import CASES
    cut = [c for c in CASES if bwd(1, *c[:5], (c[5] + 7) // 8 * 8, *c[7:]).flags & 64]
    assert len(cut) == len(CASES) - 1      # (the window of 60 and 30 leaves one step per key tile: uncut)


@pytest.mark.parametrize('call, rows', [
    ((1, 8, 2, 2048, 2048, 128), False), ((1, 8, 2, 2048, 2048, 128, True), False), ((1, 8, 2, 1024, 1024, 256), False),
    ((1, 8, 2, 1024, 1024, 64), False), ((1, 12, 12, 600, 900, 256), False), ((1, 4, 4, 2048, 2048, 256), False),
    ((1, 8, 2, 1024, 1024, 64, True), True), ((1, 2, 2, 2048, 2048, 128), True), ((1, 32, 8, 512, 512, 128, True), True),
])
def test_packed_rows_only_where_their_xcds_are_not_the_bottleneck(call, rows):
    """two K/V heads put all row blocks on two of the eight XCDs: 157 us where whole tiles take 57"""
    assert bool(fwd(*call).flags & 128) == rows


def fwd32(B, H, Sq, Sk, D, causal=False):
    from aotriton_amd.pyaotriton.v3.flash import attn_fwd_params, query_fwd_config
    x = attn_fwd_params()
    f32 = lambda *s: view(*s, name='kFloat32')
    x.Q, x.K, x.V, x.Out = f32(B, H, Sq, D), f32(B, H, Sk, D), f32(B, H, Sk, D), f32(B, H, Sq, D)
    _common(x, B, H, Sq, Sk, causal, 0.0, False)
    err, c = query_fwd_config(x, 256)
    assert int(err) == 0
    return c


@pytest.mark.parametrize('call, rows', [
    ((1, 16, 512, 512, 128), 32), ((8, 8, 512, 512, 128), 64), ((16, 8, 512, 512, 128), 64), ((8, 8, 128, 128, 128), 32),
    ((16, 8, 192, 192, 128), 64), ((24, 8, 128, 128, 128), 64), ((128, 8, 128, 128, 128), 64), ((4, 8, 1024, 1024, 128, True), 32),
    ((16, 8, 1024, 1024, 128), 64), ((16, 16, 1, 1000, 128), 32), ((128, 8, 128, 128, 64), 32), ((600, 16, 256, 256, 128), 64),
])
def test_fp32_rows_of_a_workgroup(call, rows):
    """at 128 columns the kernel that needs less of the CUs' time; always 32 rows at 64"""
    assert fwd32(*call).block_m == rows


def test_narrow_windows_leave_items_whole_where_parts_only_make_rounds():
    assert bwd(1, 1, 2, 2, 1536, 1536, 128, (200, 0), 0.1).flags & 64 == 0
    assert bwd(1, 1, 2, 2, 1536, 1536, 128, True, 0.1).flags & 64
    assert bwd(1, 1, 8, 2, 1536, 1536, 128, (200, 0), 0.1).flags & 64


@pytest.mark.parametrize('causal', [False, True, (200, 100)])
def test_a_caller_may_name_any_longest_sequence(causal):
    """the maximal lengths of packed sequences need not be those of the tensors; the choice of kernels neither grows with them nor
    fails on them"""
    lens = [5000, 3000, 9000, 3000]
    for slot, m, n in [(None, 256, 64), (1, 32, 256), (2, 256, 32)]:
        for longest in (1 << 24, 1 << 30, (1 << 31) - 200, (1 << 31) - 1):
            c = packed(slot, lens, lens, 16, 8, 128, causal, longest)
            assert (c.block_m, c.block_n) in ((m, n), (64, 128) if slot == 1 else (128, 64))


@pytest.mark.parametrize('call, rows', [
    ((5, 24, 8, 24, 108, 256), False), ((3, 24, 8, 75, 230, 256), False), ((1, 32, 8, 200, 200, 256), False), ((2, 16, 16, 200, 200, 256), False),
    ((1, 24, 8, 227, 247, 256), False), ((1, 32, 8, 64, 64, 256, True), False), ((2, 16, 16, 34, 477, 256), True), ((2, 4, 4, 209, 1204, 256), True),
    ((4, 12, 12, 51, 1968, 256), True), ((1, 8, 2, 256, 4096, 256), True), ((1, 32, 8, 1, 300, 256), True), ((6, 64, 8, 6, 6, 256, True), True),
])
def test_packed_rows_at_head_dim_256_where_they_are_sooner(call, rows):
    """us, rows / tiles: 12.5 / 10.3, 16.0 / 13.8, 15.6 / 13.9, 15.7 / 14.0, 16.1 / 15.3, 11.2 / 9.9; 17.1 / 18.7, 23.5 / 35.2, 34 / 53, 37 / 101,
    12.0 / 13.7, 10.3 / 14.5"""
    assert bool(fwd(*call).flags & 128) == rows


def _rows(Sk, start=0, apart=1):
    """strides of a (2, 4, 300, Sk) bias whose rows are `Sk + start` long and whose columns are `apart` apart"""
    row = (Sk + start) * apart
    return (4 * 300 * row, 300 * row, row, apart)


@pytest.mark.parametrize('Sk, D, bias, at, pairs', [
    (264, 256, False, 0, True), (131, 256, False, 0, True), (264, 136, False, 0, True), (264, 128, False, 0, False),
    (264, 256, _rows(264), 0, True), (264, 256, _rows(264), 16, True), (264, 200, _rows(264, 8), 0, True), (264, 256, (0, 0, 0, 1), 0, True),
    (264, 256, _rows(264), 2, False), (264, 256, _rows(264, 1), 0, False), (260, 256, _rows(260, 4), 0, False), (264, 256, _rows(264, 0, 2), 0, False),
    (264, 128, _rows(264), 0, False),
])
def test_dkdv_by_pairs_of_waves(Sk, D, bias, at, pairs):
    """head dims above 128 that store dS, without a bias or with one whose rows are whole 16-byte pieces at such places; never recomputing or for
    packed sequences"""
    from aotriton_amd._lib import lib
    shape = lambda c: (c.block_m, c.block_n, c.num_waves)
    assert (shape(bwd(1, 2, 4, 4, 300, Sk, D, bias=bias, at=at)) == (32, 128, 8)) == pairs
    lib.fa_set_bwd_workspace_limit(0)
    try:
        assert shape(bwd(1, 2, 4, 4, 300, Sk, D, bias=bias, at=at)) != (32, 128, 8)
    finally:
        lib.fa_set_bwd_workspace_limit(-1)
    if not bias:
        assert packed(1, [100, 200], [100, 200], 4, 4, D).num_waves == 4
