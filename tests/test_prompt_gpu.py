"""The prompt GEMM (more than 32 rows) against float64, at the edges of its tiles: rows around the 64/96/128-row
tiles and several row tiles, an odd strip, one group, padded quads, blocks split over K (all of them, or the
ones after the whole rounds), both scale dtypes and the three output forms; and QLinear's route to it."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def weights(N, K, dtype, seed=0):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    q = torch.randint(0, 256, (N, K // 2), dtype=torch.uint8, device="cuda", generator=g)
    s = (torch.rand(N, K // 128, device="cuda", generator=g) * 0.018 + 0.002).to(dtype)
    m = (torch.rand(N, K // 128, device="cuda", generator=g) * 0.14 - 0.15).to(dtype)
    return q, s, m


def product(x, w):
    q, s, m = w
    c = torch.stack([q & 15, q >> 4], -1).view(q.shape[0], s.shape[1], 128).double()
    return x.double() @ (c * s.double()[..., None] + m.double()[..., None]).view(q.shape[0], -1).T


def check(y, ref, what):
    # one bf16 rounding (2^-9 relative, doubled) plus the fp32 sums' noise relative to the largest output
    err = (y.double() - ref).abs()
    bound = ref.abs() * 2 ** -8 + ref.abs().max() * 2 ** -14
    assert bool((err <= bound).all()), (what, float((err - bound).max()))


@pytest.mark.parametrize("N,K", [(16, 128), (32, 384), (144, 640), (1024, 2176), (33024, 1152), (34816, 256)])
@pytest.mark.parametrize("T", [33, 64, 65, 97, 128, 129, 257])
def test_prompt_matches_float64(dev, T, N, K):
    from tokenrush_amd import gfx950
    from tokenrush_amd.fused import silu_mul
    dtype = torch.float16 if T % 2 else torch.bfloat16
    print(f"prompt T={T} N={N} K={K} {dtype}", flush=True)
    w = weights(N, K, dtype, T + N)
    x = torch.randn(T, K, device=dev).to(torch.bfloat16)
    ref = product(x, w)
    B, s, _ = gfx950.pack(*w)
    y = gfx950.mul_prompt(x, B, s)
    check(y, ref, (T, N, K))
    assert torch.equal(y, gfx950.mul_prompt(x, B, s))
    if N % 32 == 0:
        Bp, sp, _ = gfx950.pack(*w, pairs=True)
        yp = gfx950.mul_prompt(x, Bp, sp, gfx950.PROMPT_PAIRS)
        check(yp, ref, ("pairs", T, N, K))
        assert torch.equal(gfx950.mul_prompt(x, Bp, sp, gfx950.PROMPT_SILU), silu_mul(yp))


def test_prompt_rejects(dev):
    from tokenrush_amd import gfx950
    B, s, _ = gfx950.pack(*weights(32, 256, torch.bfloat16))
    x = torch.randn(64, 256, device=dev).to(torch.bfloat16)
    for bad in (x[:32], x[:, :128], x.float(), torch.randn(64, 512, device=dev).to(torch.bfloat16)[:, ::2]):
        with pytest.raises(RuntimeError):
            gfx950.mul_prompt(bad, B, s)


@pytest.mark.parametrize("layout", ["rows", "gate_up"])
def test_qlinear_prompt_route(dev, layout):
    """Every form of x that the dense path takes is still taken: strided and unaligned rows on the kernel, other
    dtypes, gradients, autocast, vmap and more dimensions on the dense path."""
    from tokenrush_amd.quant import QLinear
    w = weights(96, 640, torch.bfloat16, 3)
    lin, dense = QLinear(*w, layout=layout), QLinear(*w, backend="dequant")
    wide = torch.randn(300, 1300, device=dev).to(torch.bfloat16)
    flat = torch.randn(70 * 640 + 1, device=dev).to(torch.bfloat16)
    for x in (wide[:70, :640], wide[:70, 1:641], wide[::4, :1280:2], flat[1:].view(70, 640), wide[:256, :640]):
        check(lin(x), product(x, w), (layout, x.shape, x.stride()))
        out = torch.empty(x.shape[0], 96, dtype=torch.bfloat16, device=dev)
        assert lin(x, out=out) is out and torch.equal(out, lin(x))
    assert torch.equal(lin(wide[:257, :640]), dense(wide[:257, :640]))   # past the kernel's range
    x = wide[:70, :640].contiguous()
    for dt in (torch.float32, torch.float16):
        assert torch.equal(lin(x.to(dt)), dense(x.to(dt))) and lin(x.to(dt)).dtype == dt
    xg = x.float().requires_grad_()
    lin(xg.to(torch.bfloat16)).sum().backward()
    assert xg.grad is not None and bool((xg.grad != 0).any())
    with torch.autocast("cuda", dtype=torch.float16):
        assert lin(x).dtype == torch.float16
    assert lin(wide[:80, :640].reshape(40, 2, 640)).shape == (40, 2, 96)
    assert torch.equal(torch.vmap(lin)(x.unsqueeze(0).expand(2, 70, 640)), dense(x).expand(2, 70, 96))
    bad = x.clone()
    bad[3, 5] = float("inf")              # a bad row stays in its row
    y, ok = lin(bad), torch.arange(70, device=dev) != 3
    assert bool(torch.isfinite(y[ok]).all()) and torch.equal(y[ok], lin(x)[ok]) and not bool(torch.isfinite(y[3]).any())
