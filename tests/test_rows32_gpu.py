"""The one-slot GEMM for 17 to 32 rows and 24 < K / 128 <= 40 against float64, at its edges: the ends of the K
range, the change from four to five groups per wave, padded quads, a last wave with one group, one strip and one
strip more than a round of workgroups; rows independent of M, strips per workgroup, the fused silu; and the
K-slot sum that explicit slots still take there, call after call."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def weights(N, K, dtype, seed):
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


@pytest.mark.parametrize("K", [3200, 3712, 4096, 4224, 4608, 5120])
@pytest.mark.parametrize("N", [16, 48, 4096, 4128])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_matches_float64(dev, N, K, dtype):
    from tokenrush_amd import gfx950
    from tokenrush_amd.fused import silu_mul
    print(f"rows32 N={N} K={K} {dtype}", flush=True)
    w = weights(N, K, dtype, N + K)
    x = torch.randn(32, K, device=dev).to(torch.bfloat16)
    B, s, _ = gfx950.pack(*w)
    y = gfx950.mul(x, B, s)
    check(y, product(x, w), (N, K))
    for M in (17, 24, 31):
        assert torch.equal(gfx950.mul(x[:M].contiguous(), B, s), y[:M]), M
    for R in (1, 3, 400):
        assert torch.equal(gfx950.mul(x, B, s, strips_per_wg=R), y), R
    if N % 32 == 0:
        Bp, sp, _ = gfx950.pack(*w, pairs=True)
        assert torch.equal(gfx950.unpair(gfx950.mul(x, Bp, sp)), y)
        assert torch.equal(gfx950.mul_silu(x, Bp, sp), silu_mul(y))


@pytest.mark.parametrize("slots", [2, 3])
def test_explicit_slots_sum(dev, slots):
    from tokenrush_amd import gfx950
    w = weights(4112, 5120, torch.bfloat16, 7)
    x = torch.randn(32, 5120, device=dev).to(torch.bfloat16)
    B, s, _ = gfx950.pack(*w)
    first = gfx950.mul(x, B, s, slots=slots)
    check(first, product(x, w), slots)
    again = [gfx950.mul(x, B, s, slots=slots) for _ in range(30)]
    assert all(torch.equal(first, y) for y in again)
