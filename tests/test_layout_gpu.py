"""The conversions between the engine packing, the quad layout and dense weights, bit for bit against the
oracle, at the edges of their tiles: one strip, one group, padded and whole quads, the pair layout, a byte
tensor that starts off a 4-byte boundary, extreme parameters."""
import numpy as np
import pytest
import torch

from oracle import int4 as o

pytestmark = pytest.mark.gpu

TDT = {"bf16": torch.bfloat16, "fp16": torch.float16}


def weights(N, K, dtype, seed=0, extreme=False):
    p, s, m = o.make_weights(N, K, seed=seed, dtype=dtype)
    s, m = (torch.from_numpy(v).to(TDT[dtype]) for v in (s, m))
    if extreme:   # overflow in either rounding, infinities, NaN, zero and the smallest values
        big = torch.finfo(TDT[dtype]).max
        tiny = torch.finfo(TDT[dtype]).smallest_normal
        s.view(-1)[:6] = torch.tensor([big, 0.0, tiny, float("inf"), float("nan"), tiny / 4], dtype=TDT[dtype])
        m.view(-1)[:4] = torch.tensor([-big, big, -tiny, -float("inf")], dtype=TDT[dtype])
    return torch.from_numpy(p), s, m


def bits(t):
    return t.contiguous().view(torch.int16)


@pytest.mark.parametrize("N,K", [(16, 128), (32, 384), (48, 512), (96, 640), (1024, 2176), (34816, 256)])
@pytest.mark.parametrize("pairs", [False, True])
@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
def test_pack_unpack_dequant(dev, N, K, pairs, dtype):
    from tokenrush_amd import gfx950
    if pairs and N % 32:
        pytest.skip("pairs need N % 32 == 0")
    print(f"layout N={N} K={K} pairs={pairs} {dtype}", flush=True)
    p, s, m = weights(N, K, dtype, extreme=True)
    raw = torch.empty(p.numel() + 1, dtype=torch.uint8, device=dev)
    q = raw[1:].view(p.shape)             # off every alignment
    q.copy_(p)
    sd, md = s.to(dev), m.to(dev)
    B, sp, mp = gfx950.pack(q, sd, md, pairs=pairs)
    src = np.arange(N)
    if pairs:                             # packed strip t: gate rows 8t.., up rows N/2 + 8t..
        src = src.reshape(2, N // 16, 8).transpose(1, 0, 2).reshape(-1)
    strips = B[..., :4096].reshape(N // 16, -1, 4, 64, 4, 4).cpu().numpy()   # strip, quad, group, lane, word, byte
    codes = np.zeros((N, o.padded_groups(K) * 128), np.uint8)
    nib = np.stack([strips & 15, strips >> 4], -1).reshape(*strips.shape[:5], 8)
    for lane in range(64):
        for k in range(8):                # code 2p in nibble p, code 2p + 1 in nibble p + 4
            v = nib[:, :, :, lane, :, k // 2 + 4 * (k % 2)]
            codes[lane % 16::16].reshape(N // 16, -1, 4, 4, 32)[..., 8 * (lane // 16) + k] = v
    want = np.stack([p.numpy() & 15, p.numpy() >> 4], -1).reshape(N, K)[src]
    assert np.array_equal(codes[:, :K], want) and not codes[:, K:].any()
    q2, s2, m2 = gfx950.unpack(B, sp, mp, K, pairs=pairs)
    assert torch.equal(q, q2) and torch.equal(bits(sd), bits(s2)) and torch.equal(bits(md), bits(m2))
    dense = gfx950.dequantize(q, sd, md)
    assert torch.equal(bits(gfx950.dequantize_packed(B, sp, K, pairs)), bits(dense))
    as_bf = gfx950.dequantize_packed(B, sp, K, pairs, torch.bfloat16)
    num = ~torch.isnan(dense)
    assert torch.equal(torch.isnan(as_bf), ~num)
    assert torch.equal(bits(as_bf)[num], bits(dense.to(torch.bfloat16))[num])
    w = torch.stack([p & 15, p >> 4], -1).view(N, K // 128, 128).to(s.dtype)   # two roundings on the CPU
    ref = w.mul_(s[..., None]).add_(m[..., None]).view(N, K)
    nan = torch.isnan(ref)
    assert torch.equal(torch.isnan(dense.cpu()), nan)
    assert torch.equal(bits(dense.cpu())[~nan], bits(ref)[~nan])


@pytest.mark.parametrize("layout", ["rows", "gate_up"])
@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
def test_qlinear_dense_forms(dev, layout, dtype):
    from tokenrush_amd.quant import QLinear
    p, s, m = (t.to(dev) for t in weights(64, 640, dtype, seed=3))
    a, b = QLinear(p, s, m, layout=layout), QLinear(p, s, m, backend="dequant")
    assert a.dequantize().dtype == s.dtype and torch.equal(a.dequantize(), b.dequantize())
    for dt in (torch.bfloat16, torch.float16, torch.float32):
        assert torch.equal(a.dequantize(dt), b.dequantize().to(dt)) and a.dequantize(dt).dtype == dt
