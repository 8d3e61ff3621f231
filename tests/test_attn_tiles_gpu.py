"""The flash-decoding split kernel at the edges of its tiles against float64: query rows of one to three 16-row
tiles and of several row groups, key counts around the 32-key block and the four-block round, few and many
splits, chains and trees, and keys that outgrow a row's first maximum by more than the kernel's restart
threshold."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


def exact(q, u, k, ks, v, vs, pos, sees, HQ, HKV):
    M, G = q.shape[0], HQ // HKV
    q = q.double().view(M, HQ, 256)
    gate = torch.sigmoid(u[:, :HQ * 512].double().view(M, HQ, 2, 256)[:, :, 1])
    y = torch.empty(M, HQ, 256, dtype=torch.float64, device=q.device)
    for h in range(HQ):
        j = h // G
        K = k[j, :pos + M].double() * ks[j, :pos + M, None].double()
        V = v[j, :pos + M].double() * vs[j, :pos + M, None].double()
        s = q[:, h] @ K.T / 16.0
        s[:, pos:] = s[:, pos:].masked_fill(~sees, -math.inf)
        y[:, h] = torch.softmax(s, -1) @ V
    return (y * gate).reshape(M, -1)


def run(dev, M, HQ, HKV, pos, tree, nsplit, seed=0, spikes=False):
    from tokenrush_amd.attn import AttnConfig, attn_decode_fused
    print(f"attn M={M} heads={HQ}/{HKV} pos={pos} tree={tree} nsplit={nsplit} spikes={spikes}", flush=True)
    g = torch.Generator(device=dev)
    g.manual_seed(seed)
    L = pos + M + 5
    k, v = (torch.randn(HKV, L, 256, device=dev, generator=g) for _ in range(2))
    if spikes:   # scores climb by hundreds of log2 units along the keys, and a last key far below
        k *= torch.linspace(0.2, 40, L, device=dev)[None, :, None]
        k[:, -1] *= 0.01
    ks, vs = (t.abs().amax(-1) / 448 for t in (k, v))
    k, v = ((t / s[..., None]).to(torch.float8_e4m3fn) for t, s in ((k, ks), (v, vs)))
    q = torch.randn(M, HQ * 256, device=dev, generator=g).to(torch.bfloat16)
    u = torch.randn(M, HQ * 512 + HKV * 512, device=dev, generator=g).to(torch.bfloat16)
    parent = [0] + [max(0, (i - 1) // 2) for i in range(1, M)] if tree else [max(0, i - 1) for i in range(M)]
    sees = torch.zeros(M, M, dtype=torch.bool, device=dev)
    for t in range(M):
        n = t
        while True:
            sees[t, n] = True
            if n == 0:
                break
            n = parent[n]
    par = torch.tensor(parent, dtype=torch.int32, device=dev) if tree else None
    cfg = AttnConfig(HQ, HKV, 256, 64, 1e7, 1e-6)
    args = (q, u, k, v, torch.tensor([pos], device=dev), cfg, ks, vs)
    y = attn_decode_fused(*args, NSPLIT=nsplit, parent=par)
    assert torch.equal(y, attn_decode_fused(*args, NSPLIT=nsplit, parent=par))
    ref = exact(q, u, k, ks, v, vs, pos, sees, HQ, HKV)
    err = (y.double() - ref).norm() / ref.norm()
    # bf16 probabilities, output and gate: 2^-9 each in the root mean square, three of them
    assert err < 5e-3, float(err)


@pytest.mark.parametrize("M,HQ,HKV", [(1, 2, 1), (8, 2, 1), (3, 24, 4), (5, 24, 4), (8, 24, 4), (8, 8, 1), (1, 40, 40)])
@pytest.mark.parametrize("pos", [0, 1, 24, 31, 33, 120, 129, 1000])
def test_chain_rows_and_keys(dev, M, HQ, HKV, pos):
    run(dev, M, HQ, HKV, pos, False, None, seed=pos + M)


@pytest.mark.parametrize("M,HQ,HKV", [(2, 24, 4), (9, 24, 4), (17, 24, 4), (32, 24, 4), (32, 8, 1), (32, 2, 1)])
@pytest.mark.parametrize("pos", [0, 100, 2000])
def test_tree_row_groups(dev, M, HQ, HKV, pos):
    run(dev, M, HQ, HKV, pos, True, None, seed=pos + M)


@pytest.mark.parametrize("nsplit", [1, 3, 64, 256])
@pytest.mark.parametrize("tree", [False, True])
def test_split_counts(dev, nsplit, tree):
    run(dev, 8, 6, 1, 3000, tree, nsplit)


@pytest.mark.parametrize("nsplit", [1, 5, 64])
def test_growing_scores(dev, nsplit):
    run(dev, 8, 6, 1, 1500, False, nsplit, spikes=True)
    run(dev, 20, 6, 1, 700, True, nsplit, spikes=True)


@pytest.mark.parametrize("M", [1, 5, 8])
@pytest.mark.parametrize("pos", [503, 504, 511, 512, 1016, 1023, 1024, 1030])
@pytest.mark.parametrize("spikes", [False, True])
def test_rounds_per_split(dev, M, pos, spikes):
    """Four splits of one, two and three rounds of four blocks, one to three query tiles."""
    run(dev, M, 6, 1, pos, False, 4, seed=pos, spikes=spikes)
