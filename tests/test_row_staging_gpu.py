"""The verify GEMM at 1 to 16 rows: x staged through LDS beside the reduction ring and inside it, or read directly,
with one strip and two in flight."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sdt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("N,K,slots", [
    (16, 128, None),      # one strip, one wave, three padding groups; at 9 to 16 rows x read directly
    (48, 640, None),      # two waves, the second with one group; likewise
    (8208, 640, None),    # 513 strips: staged again
    (12304, 3456, None),  # seven waves, four strips per workgroup: two in flight up to 8 rows
    (4112, 2048, None),   # 257 strips: one workgroup has two, three workgroups to a CU
    (528, 6144, 1),       # twelve waves
    (272, 17408, 3),      # 34 blocks over three slots: waves without a block
])
def test_row_ranges(dev, N, K, slots, sdt):
    """Each row of every call of 1 to 16 rows has the bits it has at 16, and the partials' sum is within
    fp32's bound of float64: per output a chain of at most 128 products, K / 128 folds and the slots,
    each rounding relative to the magnitudes added (codes carry an offset of 128 that the min term removes)."""
    from tokenrush_amd import gfx950
    g = torch.Generator().manual_seed(N + K)
    q = torch.randint(0, 256, (N, K // 2), dtype=torch.uint8, generator=g)
    s = (torch.rand(N, K // 128, generator=g) * 0.018 + 0.002).to(sdt)
    mn = (torch.rand(N, K // 128, generator=g) * 0.14 - 0.15).to(sdt)
    x = torch.randn(16, K, generator=g).bfloat16()
    B, sm = gfx950.pack(q.cuda(), s.cuda(), mn.cuda())[:2]
    codes = torch.stack([q & 15, q >> 4], -1).view(N, K // 128, 128).double()
    xd = x.double()
    want = xd @ (codes * s.double()[..., None] + mn.double()[..., None]).view(N, K).T
    size = torch.einsum("mgk,ng->mn", xd.abs().view(16, -1, 128), 143 * s.double() + (mn.double() - 128 * s.double()).abs())
    bound = (128 + K // 128 + 16) * 2.0**-23 * size
    xg = x.cuda()
    full, part16 = gfx950.mul(xg, B, sm), gfx950.mul_partial(xg, B, sm, n_slots=slots)
    assert (part16.double().sum(0).cpu() - want).abs().le(bound).all()
    for M in (1, 2, 7, 8, 9, 10, 15):
        xm = xg[:M].contiguous()
        assert torch.equal(gfx950.mul(xm, B, sm), full[:M]), M
        assert torch.equal(gfx950.mul_partial(xm, B, sm, n_slots=slots if slots else part16.shape[0]), part16[:, :M]), M
