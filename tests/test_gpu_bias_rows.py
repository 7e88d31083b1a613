"""Forward with a bias whose rows start anywhere (odd lengths) and end inside a key tile: against a computation in 64 bits,
at the edges of the pieces and tiles, the bias filling its memory to the last byte with NaN in front of it."""
import pytest
import torch

from test_launch_queries import fwd

BF, HF = torch.bfloat16, torch.float16
CASES = [
    # B, H, Sq, Sk, D, dtype, causal, dropout
    (8, 12, 513, 513, 64, BF, False),
    (2, 3, 70, 131, 64, HF, False),
    (2, 3, 300, 513, 64, HF, True),
    (1, 2, 129, 9, 64, BF, False),
    (1, 2, 40, 8, 64, HF, False),
    (1, 2, 40, 7, 64, HF, False),           # no piece fits: element by element
    (4, 16, 203, 255, 40, BF, True),
    (16, 32, 300, 97, 64, HF, (50, 3)),
    (4, 8, 260, 383, 128, HF, True),
    (1, 2, 200, 65, 80, BF, False),
    (2, 4, 300, 191, 128, BF, (-20, 90)),
    (2, 4, 300, 261, 256, BF, (100, 0)),
    (1, 3, 260, 389, 256, HF, True),
    (1, 2, 140, 97, 200, BF, False),
    (1, 2, 129, 32, 256, HF, False),
    (1, 2, 40, 7, 256, BF, False),
    (4, 16, 290, 300, 64, HF, (100, 3)),     # whole tiles, waves with few rows or none
    (4, 16, 270, 392, 64, BF, (200, 10)),
    (4, 16, 270, 392, 96, BF, True),
    (4, 16, 257, 256, 128, HF, True),
]


def _id(c):
    return '-'.join(str(x).replace('torch.', '') for x in c)


def test_a_row_bias_takes_small_tiles():
    assert fwd(8, 12, 12, 513, 513, 64, False, 0.0, True).block_m == 128
    assert fwd(8, 12, 12, 520, 520, 64, False, 0.0, True).block_m == 128
    assert fwd(8, 12, 12, 2048, 2048, 64, False, 0.0, True).block_m == 256


@pytest.mark.gpu
@pytest.mark.parametrize('p', [0.0, 0.2])
@pytest.mark.parametrize('case', CASES, ids=_id)
def test_bias_rows_at_any_alignment(case, p):
    from aotriton_amd import flash
    B, H, Sq, Sk, D, dt, causal = case
    g = torch.Generator(device='cuda').manual_seed(2)
    rn = lambda *s: torch.randn(*s, device='cuda', generator=g).to(dt)
    q, k, v = rn(B, H, Sq, D), rn(B, H, Sk, D), rn(B, H, Sk, D)
    room = torch.full((B * H * Sq * Sk + 1,), float('nan'), device='cuda', dtype=dt)
    odd = room[1:].view(B, H, Sq, Sk).copy_(rn(B, H, Sq, Sk))
    wide = torch.full((B, H, Sq, (Sk + 7) // 8 * 8), float('nan'), device='cuda', dtype=dt)
    wide[..., :Sk] = odd
    seed, off = (torch.tensor([x], device='cuda', dtype=torch.uint64) for x in (3, 4))
    null, out = torch.empty([0], device='cuda', dtype=torch.uint64), []
    for b in (odd, wide[..., :Sk]):
        o, L = torch.empty_like(q), torch.empty(B * H, Sq, device='cuda')
        assert flash.attn_fwd(q, k, v, b, D ** -0.5, L, o, p, seed, off, 0, null, null, None, causal, null) == flash.hipError_t.hipSuccess
        out.append((o, L))
    s = torch.matmul(q.double(), k.double().transpose(-1, -2).contiguous()) * D ** -0.5 + odd.double()
    if causal:
        left, right = (Sq, 0) if causal is True else causal
        m, n = torch.arange(Sq, device='cuda')[:, None], torch.arange(Sk, device='cuda')
        s = s.masked_fill((n < m - left) | (n > m + right), float('-inf'))
    lse = torch.logsumexp(s, -1).view(B * H, Sq)
    seen = lse > float('-inf')
    for o, L in out:
        assert ((L - lse)[seen].abs() < 1e-5 * (1 + lse[seen].abs())).all()
        assert torch.isfinite(o).all()
    if p:      # the same mask on both: the results differ by the roundings of P only
        d = (out[0][0].double() - out[1][0].double()).norm() / out[1][0].double().norm().clamp_min(1e-30)
        assert d.item() < 2 * torch.finfo(dt).eps
    else:
        want = torch.matmul(torch.softmax(s, -1).nan_to_num(0.0), v.double())
        for o, _ in out:      # P rounded, the result rounded
            assert ((o.double() - want).norm() / want.norm()).item() < 3 * torch.finfo(dt).eps / 2


@pytest.mark.gpu
@pytest.mark.parametrize('p', [0.0, 0.2])
@pytest.mark.parametrize('step', [(1 << 21) - 1, 1 << 21])
def test_rows_far_apart(step, p):
    """Rows of the bias as far apart as they may be (their offsets are kept in 32 bits), next to the same rows close together."""
    from aotriton_amd import flash
    B, H, Sq, Sk, D, dt = 8, 16, 262, 136, 128, HF
    assert fwd(B, H, H, Sq, Sk, D, False, p, True).block_m == 256
    g = torch.Generator(device='cuda').manual_seed(5)
    rn = lambda *s: torch.randn(*s, device='cuda', generator=g).to(dt)
    q, k, v, near = rn(B, H, Sq, D), rn(B, H, Sk, D), rn(B, H, Sk, D), rn(Sq, Sk)
    far = torch.empty((Sq - 1) * step + Sk, device='cuda', dtype=dt).as_strided((Sq, Sk), (step, 1)).copy_(near)
    seed, off = (torch.tensor([x], device='cuda', dtype=torch.uint64) for x in (3, 4))
    null, out = torch.empty([0], device='cuda', dtype=torch.uint64), []
    for b in (near, far):
        o, L = torch.empty_like(q), torch.empty(B * H, Sq, device='cuda')
        b = b.expand(B, H, Sq, Sk)
        assert flash.attn_fwd(q, k, v, b, D ** -0.5, L, o, p, seed, off, 0, null, null, None, False, null) == flash.hipError_t.hipSuccess
        out.append((o, L))
    assert (out[0][1] - out[1][1]).abs().max().item() < 1e-5 * (1 + out[0][1].abs().max().item())
    d = (out[0][0].double() - out[1][0].double()).norm() / out[0][0].double().norm()
    assert d.item() < 2 * torch.finfo(dt).eps


@pytest.mark.gpu
@pytest.mark.parametrize('p', [0.0, 0.2])
@pytest.mark.parametrize('D,dt,causal', [(64, HF, True), (64, BF, False), (96, BF, True), (128, BF, True), (128, HF, (90, 20))])
def test_rows_that_overlap(D, dt, causal, p):
    """Rows that start 16 bytes apart in one vector of memory (a bias by distance), the last of them ending where the memory does, and
    the same rows apart: the same bits."""
    from aotriton_amd import flash
    B, H, Sq, Sk = 4, 16, 291, 384
    assert fwd(B, H, H, Sq, Sk, D, causal, 0.2, True).block_m == 256
    g = torch.Generator(device='cuda').manual_seed(6)
    rn = lambda *s: torch.randn(*s, device='cuda', generator=g).to(dt)
    q, k, v = rn(B, H, Sq, D), rn(B, H, Sk, D), rn(B, H, Sk, D)
    n = 8 * (Sq - 1) + Sk
    memory = torch.full((H * n + 64,), float('nan'), device='cuda', dtype=dt)
    memory[:H * n] = rn(H * n)
    near = memory.as_strided((B, H, Sq, Sk), (0, n, 8, 1))
    seed, off = (torch.tensor([x], device='cuda', dtype=torch.uint64) for x in (3, 4))
    null, out = torch.empty([0], device='cuda', dtype=torch.uint64), []
    for b in (near, near.contiguous()):
        o, L = torch.empty_like(q), torch.empty(B * H, Sq, device='cuda')
        assert flash.attn_fwd(q, k, v, b, D ** -0.5, L, o, p, seed, off, 0, null, null, None, causal, null) == flash.hipError_t.hipSuccess
        out.append((o, L))
    assert torch.isfinite(out[0][0]).all()
    assert torch.equal(out[0][0], out[1][0]) and torch.equal(out[0][1], out[1][1])
