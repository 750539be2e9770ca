"""GPU parity of the shared-x perturbed linear (config 2) against oracle.model.lowrank_sumsq.

Both evaluations of the per-member sums of squares (the expanded square on the MFMA units, and every element formed)
are checked against the float64 oracle. Tolerances: S_i within 1e-4 relative at the reduced shapes (bf16 operands,
fp32 accumulation; the roundings of x W^T and x . b agree with the oracle's except in rare last-bit ties); at the full
config-2 size the error must also stay within 1e-2 of S_i's member-specific part S_i - sum (x W^T)^2, which at
sigma 1e-3 is about 0.2% of S_i (so a wrong rank-1 term fails even though S_i barely moves)."""
import pytest
import torch

from oracle import model as om

pytestmark = pytest.mark.gpu


def _inputs(T, n_in, n_out, m, seed, a_off=7, gap=3):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(T, n_in, generator=g).bfloat16()
    W = (torch.randn(n_out, n_in, generator=g) * 0.02).bfloat16()
    stride = a_off + n_out + gap + n_in + 5
    rows = torch.randn(m, stride, generator=g)
    b_off = a_off + n_out + gap
    a, b = rows[:, a_off:a_off + n_out], rows[:, b_off:b_off + n_in]
    return x, W, rows, a_off, b_off, a, b


@pytest.mark.parametrize('mode', ['expansion', 'direct'])
def test_shared_sumsq_small(dev, mode):
    """m = 40 (a padded second member tile), 2 x 2 output tiles, sigma large enough that the rank-1 term dominates."""
    from noise_amd.population import lowrank_sumsq
    T, n_in, n_out, m = 512, 64, 512, 40
    print(f'lowrank shared {mode} T={T} in={n_in} out={n_out} m={m}', flush=True)
    x, W, rows, a_off, b_off, a, b = _inputs(T, n_in, n_out, m, seed=1)
    sign = torch.tensor([0.05 if i % 2 == 0 else -0.05 for i in range(m)])
    sign[5] = 0.0
    want, c2 = om.lowrank_sumsq(x.float(), W.float(), a, b, sign)
    got = lowrank_sumsq(x.to(dev), W.to(dev), rows.to(dev), a_off, b_off, sign.to(dev), mode=mode).cpu().double()
    rel = ((got - want).abs() / want.abs()).max().item()
    assert rel < 1e-4, rel
    assert abs(got[5] - c2) / c2 < 1e-5  # sign 0: the unperturbed sum of squares


def test_shared_modes_agree_and_y(dev):
    """With y stored, every element equals the oracle's c + (s u) a; the two evaluations give the same sums."""
    from noise_amd.population import lowrank, lowrank_sumsq
    T, n_in, n_out, m = 256, 96, 256, 3
    print(f'lowrank shared y T={T} in={n_in} out={n_out} m={m}', flush=True)
    x, W, rows, a_off, b_off, a, b = _inputs(T, n_in, n_out, m, seed=2)
    sign = torch.tensor([0.1, -0.1, 0.03])
    y = lowrank(x.to(dev), W.to(dev), a.to(dev), b.to(dev), sign.to(dev)).cpu().double()
    c = (x.float() @ W.float().t()).bfloat16().double()
    u = (x.float() @ b.bfloat16().float().t()).bfloat16().double()
    ref = c[None] + (sign.double()[:, None] * u.t())[:, :, None] * a.bfloat16().double()[:, None, :]
    # a last-bit tie of the bf16 rounding of x W^T or x . b may go the other way: one bf16 step of c or of the
    # rank-1 term at most, and only in rare elements (a tie in u moves one row of one member)
    err = (y - ref).abs()
    rank1 = ref - c[None]
    assert (err <= 2.0 ** -7 * (c.abs()[None] + rank1.abs()) + 1e-5).all(), err.max().item()
    assert (err > 1e-5).float().mean().item() < 2e-2
    s1 = lowrank_sumsq(x.to(dev), W.to(dev), rows.to(dev), a_off, b_off, sign.to(dev), mode='expansion').cpu()
    s2 = lowrank_sumsq(x.to(dev), W.to(dev), rows.to(dev), a_off, b_off, sign.to(dev), mode='direct').cpu()
    assert ((s1 - s2).abs() / s2.abs()).max().item() < 1e-5
    assert ((s2.double() - (y * y).sum((1, 2))).abs() / s2.double()).max().item() < 1e-5


def test_shared_gemm_is_the_same_bits_for_32_and_64_deep_k_steps(dev):
    """in = 512 takes the GEMM with 64-deep K steps (two LDS stages), in = 544 -- the same x and W with 32 zero
    columns appended -- the one with 32-deep steps (four stages): the same 16-deep MFMA products in the same order,
    plus exact zeros, so x W^T comes out with the same bits. (The signs are 0: the rank-1 term's x . b is summed by
    another kernel whose order depends on the width.)"""
    from noise_amd.population import lowrank
    T, n_in, n_out, m, pad = 512, 512, 512, 2, 32
    print(f'lowrank shared BK64 vs BK32 T={T} in={n_in}+{pad} out={n_out}', flush=True)
    x, W, rows, a_off, b_off, a, b = _inputs(T, n_in, n_out, m, seed=4)
    sign = torch.zeros(m)
    zx, zw = torch.zeros(T, pad, dtype=torch.bfloat16), torch.zeros(n_out, pad, dtype=torch.bfloat16)
    y64 = lowrank(x.to(dev), W.to(dev), a.to(dev), b.to(dev), sign.to(dev))
    y32 = lowrank(torch.cat([x, zx], 1).to(dev), torch.cat([W, zw], 1).to(dev), a.to(dev),
                  torch.cat([b, torch.zeros(m, pad)], 1).to(dev), sign.to(dev))
    torch.cuda.synchronize()
    assert torch.equal(y64, y32)
    c = (x.float() @ W.float().t()).bfloat16()
    assert ((y64[0].float().cpu() - c.float()).abs() <= 2.0 ** -7 * c.float().abs() + 1e-6).all()


def test_shared_sumsq_config2(dev):
    """Config 2 at full size: X [32768, 512], W [2048, 512] N(0, 0.02), 64 members, sigma 1e-3; members 0 and 37
    against the float64 oracle, every member's two evaluations against each other."""
    from noise_amd.population import lowrank_sumsq
    T, n_in, n_out, m, sigma = 32768, 512, 2048, 64, 1e-3
    print(f'lowrank shared config 2 T={T} in={n_in} out={n_out} m={m}', flush=True)
    x, W, rows, a_off, b_off, a, b = _inputs(T, n_in, n_out, m, seed=3, a_off=0, gap=0)
    sign = torch.tensor([sigma if i % 2 == 0 else -sigma for i in range(m)])
    got = {md: lowrank_sumsq(x.to(dev), W.to(dev), rows.to(dev), a_off, b_off, sign.to(dev), mode=md).cpu().double()
           for md in ('expansion', 'direct')}
    assert ((got['expansion'] - got['direct']).abs() / got['direct']).max().item() < 1e-5
    pick = [0, 37]
    want, c2 = om.lowrank_sumsq(x.float(), W.float(), a, b, sign, members=pick)
    for md, s in got.items():
        for j, i in enumerate(pick):
            part = (want[j] - c2).abs().item()
            err = (s[i] - want[j]).abs().item()
            print(f'{md} member {i}: S {s[i].item():.6e} oracle {want[j].item():.6e} member part {part:.4e} '
                  f'err {err:.3e}', flush=True)
            assert err < 1e-3 * part, (md, i, err, part)  # measured 2.4e-5 of the member part


@pytest.mark.parametrize('m,T,n_in,n_out', [
    (1, 128, 32, 256),     # the smallest: one tile, one K step
    (3, 128, 544, 512),    # K not a multiple of 64 nor of a wave's 512 channels
    (5, 384, 1056, 256),   # more than one pass over the channels
    (131, 128, 64, 4096),  # past four rounds of 256 x 256 tiles: 64-deep steps; 128 rows past a 256-row tile
    (131, 128, 96, 4096),  # the same with K not a multiple of 64
])
def test_per_member_lowrank_over_its_tiles(dev, m, T, n_in, n_out):
    """The per-member perturbed linear on each of its tiles, against float64 of the same bf16 operands: the output is the
    bf16-rounded product (2^-8 of it) plus a rank-1 term whose dot is rounded to bf16 too."""
    print(f'lowrank m={m} T={T} {n_in}->{n_out}', flush=True)
    from noise_amd.population import lowrank
    g = torch.Generator(device=dev).manual_seed(m * T + n_in)
    x = torch.randn(m, T, n_in, device=dev, generator=g).bfloat16()
    w = torch.randn(n_out, n_in, device=dev, generator=g).bfloat16()
    a, b = torch.randn(m, n_out, device=dev, generator=g), torch.randn(m, n_in, device=dev, generator=g)
    sign = torch.where(torch.arange(m, device=dev) % 2 == 0, 0.5, -0.5).float()
    y = lowrank(x, w, a, b, sign)
    assert torch.isfinite(y).all()
    for i in sorted({0, 1, m // 2, m - 2, m - 1} & set(range(m))):
        xi, ai, bi = x[i].double(), a[i].bfloat16().double(), b[i].bfloat16().double()
        c, u = xi @ w.double().t(), xi @ bi
        want = c + float(sign[i]) * u[:, None] * ai
        bound = 2.0 ** -8 * (c.abs() + 0.5 * u.abs()[:, None] * ai.abs()) \
            + 2.0 ** -20 * (xi.abs() @ w.double().abs().t() + 0.5 * (xi.abs() @ bi.abs())[:, None] * ai.abs())
        assert ((y[i].double() - want).abs() <= bound).all(), i


@pytest.mark.parametrize('T,n_in,n_out,m', [
    (256, 32, 256, 1),      # the smallest; one member, so one split
    (512, 64, 512, 130),    # a split of several members; y too
    (8192, 64, 512, 130),   # two splits of 65 members: more than one LDS chunk of 64
    (32768, 32, 256, 3),    # the largest on half tiles, in either form
    (33024, 32, 256, 3),    # 256 rows more: whole tiles
    (16896, 96, 512, 5),    # the expansion on whole tiles, the per-element form on half ones
])
def test_shared_tiles_and_member_splits(dev, T, n_in, n_out, m):
    """Sums of squares on either side of the shared-x launches' rules against float64 of the bf16 operands, to the 1e-4 of
    this file (ties of the bf16 roundings); the stored y, where it is small, against its own sums."""
    from noise_amd.population import lowrank, lowrank_sumsq
    print(f'lowrank shared T={T} in={n_in} out={n_out} m={m}', flush=True)
    x, W, rows, a_off, b_off, a, b = (t.to(dev) if torch.is_tensor(t) else t for t in _inputs(T, n_in, n_out, m, seed=T + m))
    sign = torch.where(torch.arange(m, device=dev) % 2 == 0, 0.05, -0.05).float()
    c = (x.double() @ W.double().t()).bfloat16().double()
    u = (x.double() @ b.bfloat16().double().t()).bfloat16().double()
    ab = a.bfloat16().double()
    want = torch.stack([((c + float(sign[i]) * u[:, i:i + 1] * ab[i]) ** 2).sum() for i in range(m)])
    for mode in ('expansion', 'direct'):
        got = lowrank_sumsq(x, W, rows, a_off, b_off, sign, mode=mode).double()
        assert ((got - want).abs() / want).max().item() < 1e-4, mode
    if T <= 512:
        y = lowrank(x, W, a.contiguous(), b.contiguous(), sign).double()
        assert (((y * y).sum((1, 2)) - want).abs() / want).max().item() < 1e-4


@pytest.mark.parametrize('T,n_in,n_out,m', [
    (256, 128, 256, 1),    # the smallest: two K steps, fewer than the stages; one member of its tile of 32
    (512, 256, 256, 33),   # as many steps as stages; a second tile of one member
    (768, 640, 512, 96),   # three member tiles
    (1024, 2048, 256, 40),
])
def test_member_dots_are_the_same_bits_staged_or_from_memory(dev, T, n_in, n_out, m):
    """x . b of a width in 128-column steps runs as a GEMM through LDS, of other widths straight from memory: 32 columns of
    zeros more change the route and add exact zeros to every product, so every sum of squares keeps its bits."""
    from noise_amd.population import lowrank_sumsq
    print(f'lowrank shared dots T={T} in={n_in} out={n_out} m={m}', flush=True)
    x, W, rows, a_off, b_off, a, b = (t.to(dev) if torch.is_tensor(t) else t for t in _inputs(T, n_in, n_out, m, seed=T + m))
    sign = torch.where(torch.arange(m, device=dev) % 2 == 0, 0.5, -0.5).float()
    wide = [torch.nn.functional.pad(t, (0, 32)).contiguous() for t in (x, W, b)]
    wide_rows = torch.cat([a, wide[2]], 1).contiguous()
    u = x.double() @ b.bfloat16().double().t()
    assert u.abs().mean().item() > 1  # the members' terms are no small part of the sums
    for mode in ('expansion', 'direct'):
        got = lowrank_sumsq(x, W, rows, a_off, b_off, sign, mode=mode)
        want = lowrank_sumsq(wide[0], wide[1], wide_rows, 0, n_out, sign, mode=mode)
        assert torch.isfinite(got).all() and torch.equal(got, want), mode
