"""The work a user of this framework has it do, as cases that can be timed and checked.

A verify engine runs its step as one captured hipGraph, so the decode cases capture their launches
in `prepare` and `run` replays them; prompts (more than 32 rows, whose length changes from call to
call) and the weight conversion at load run eagerly. Sizes are the 64-layer hybrid's (hidden 5120,
MLP 17408, vocab 248320, 24 / 4 attention heads, 16 / 48 GDN heads), the small test model's, and
ragged ones between.

Each kind of case has make(case, seed) for its raw inputs (plain tensors, from the seed alone),
prepare, run, and an exact() in float64 from the same raw inputs without this repository's code.
"""
import math
import os
import random
import sys

import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "token-rush_amd"))

DEV = "cuda:0"
EPS = 1e-6
BF, F32, F64 = torch.bfloat16, torch.float32, torch.float64
RING = 16


def listed():
    return [
        # one token through square projections (the draft-free decode, latency bound)
        {"name": "gemv_m1", "kind": "proj", "layers": 24, "m": 1, "n": 5120, "k": 5120, "scale": "fp16"},
        # the projections and norms of one layer at the usual verify width: 1 committed token + 7 drafts
        {"name": "layer_m8", "kind": "layer", "layers": 2, "m": 8, "hidden": 5120, "qkv": 7168, "attn": 6144,
         "mlp": 17408, "scale": "fp16"},
        # the same under a 32-node draft tree, in the engine's bf16 scales
        {"name": "layer_m32", "kind": "layer", "layers": 2, "m": 32, "hidden": 5120, "qkv": 14336, "attn": 6144,
         "mlp": 17408, "scale": "bf16"},
        # the MLP on a short prompt (or the new turn of a chat) and on a long, ragged prompt chunk
        {"name": "mlp_t100", "kind": "mlp", "t": 100, "hidden": 5120, "mlp": 17408},
        {"name": "mlp_t2000", "kind": "mlp", "t": 2000, "hidden": 5120, "mlp": 17408},
        # the recurrent mixers of a chain step
        {"name": "gdn_m8", "kind": "gdn", "layers": 4, "m": 8, "tree": False, "hidden": 5120, "h": 16, "hv": 48,
         "pos": 8192},
        # ... and of a 32-node draft tree
        {"name": "gdn_tree32", "kind": "gdn", "layers": 2, "m": 32, "tree": True, "hidden": 5120, "h": 16, "hv": 48,
         "pos": 8191},
        # the attention layers of a step at 8k live tokens, and one of a long context
        {"name": "attn_m8_8k", "kind": "attn", "layers": 8, "m": 8, "tree": False, "hq": 24, "hkv": 4, "ctx": 8192},
        {"name": "attn_m4_100k", "kind": "attn", "layers": 1, "m": 4, "tree": False, "hq": 24, "hkv": 4,
         "ctx": 100001},
        # the sampled verify accept over the full vocabulary
        {"name": "accept_m8", "kind": "accept", "rule": "sampled", "m": 8, "v": 248320},
        # loading one gate/up matrix: conversion to the kernel layout, back (to save it) and to a dense matrix
        {"name": "load_gate_up", "kind": "load", "n": 34816, "k": 5120, "layout": "gate_up"},
        # a whole tree-verify step through one period of the hybrid (3 GDN + 1 attention layers) and the lm_head
        {"name": "step_tree32", "kind": "step", "m": 32, "tree": True, "hidden": 5120, "mlp": 17408, "vocab": 248320,
         "ctx": 8192},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng: random.Random):
    kind = rng.choice(["proj", "layer", "layer", "mlp", "gdn", "attn", "accept", "load", "step"])
    tree = rng.random() < 0.5
    m = rng.randint(2, 32) if tree else rng.randint(1, 8)
    c = {"kind": kind}
    if kind == "proj":
        c.update(layers=rng.randint(4, 16), m=rng.randint(1, 32), n=16 * _log(rng, 32, 768), k=128 * _log(rng, 4, 96),
                 scale=rng.choice(["fp16", "bf16"]))
    elif kind == "layer":
        hidden = 128 * rng.randint(8, 40)
        c.update(layers=2, m=rng.randint(1, 32), hidden=hidden, qkv=16 * rng.randint(64, 896),
                 attn=128 * rng.randint(8, 48), mlp=128 * rng.randint(16, 136), scale=rng.choice(["fp16", "bf16"]))
    elif kind == "mlp":
        c.update(t=_log(rng, 33, 2000), hidden=128 * rng.randint(8, 40), mlp=128 * rng.randint(16, 136))
    elif kind == "gdn":
        h, hv = rng.choice([(16, 48), (16, 48), (2, 4), (16, 32)])
        c.update(layers=rng.randint(1, 3), m=m, tree=tree, hidden=128 * rng.randint(8, 40), h=h, hv=hv,
                 pos=_log(rng, 4, 100000))
    elif kind == "attn":
        hq, hkv = rng.choice([(24, 4), (24, 4), (2, 1), (16, 4)])
        ctx = _log(rng, 64, 100000)
        c.update(layers=max(1, min(8, 65536 // ctx)), m=m, tree=tree, hq=hq, hkv=hkv, ctx=ctx)
    elif kind == "accept":
        rule = rng.choice(["greedy", "sampled", "residual", "tree"])
        m = rng.randint(2, 32) if rule == "tree" else rng.randint(2, 8)
        c.update(rule=rule, m=m, v=_log(rng, 4096, 248320))
    elif kind == "load":
        c.update(n=32 * _log(rng, 32, 1088), k=128 * _log(rng, 4, 40), layout=rng.choice(["rows", "gate_up"]))
    else:
        c.update(m=m, tree=tree, hidden=128 * rng.randint(8, 40), mlp=128 * rng.randint(16, 136),
                 vocab=16 * _log(rng, 256, 15520), ctx=_log(rng, 64, 16384))
    return c


# ------------------------------------------------------------------ raw inputs

def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _randn(g, *shape, std=1.0, mean=0.0, dtype=BF):
    return (torch.randn(*shape, device=DEV, generator=g) * std + mean).to(dtype)


def _weight(g, n, k, scale="bf16"):
    """Engine-packed int4 weight: codes uniform, scale ~U(0.002, 0.02), min ~U(-0.15, -0.01)."""
    dt = torch.float16 if scale == "fp16" else BF
    q = torch.randint(0, 256, (n, k // 2), dtype=torch.uint8, device=DEV, generator=g)
    s = (torch.rand(n, k // 128, device=DEV, generator=g) * 0.018 + 0.002).to(dt)
    mn = (torch.rand(n, k // 128, device=DEV, generator=g) * 0.14 - 0.15).to(dt)
    return q, s, mn


def _tree(m, seed):
    """parent of each node (node 0 the root, -1): at most 4 children and depth 7, as a draft tree has."""
    rng = random.Random(seed)
    parent, depth, kids = [-1], [0], [0]
    for i in range(1, m):
        j = rng.choice([j for j in range(i) if kids[j] < 4 and depth[j] < 7])
        parent.append(j)
        depth.append(depth[j] + 1)
        kids.append(0)
        kids[j] += 1
    return parent


def _parents(case, seed):
    return _tree(case["m"], seed) if case["tree"] else list(range(-1, case["m"] - 1))


def _cache(g, planes, hkv, maxlen, live, d=256):
    """FP8 K and V caches as the prep writes them (per-row scale amax / 448), rows past `live` zero."""
    out = []
    for _ in range(2):
        codes = torch.zeros(planes, hkv, maxlen, d, dtype=torch.float8_e4m3fn, device=DEV)
        scale = torch.zeros(planes, hkv, maxlen, device=DEV)
        for p in range(planes):
            x = torch.randn(hkv, live, d, device=DEV, generator=g)
            x *= torch.exp(0.3 * torch.randn(hkv, live, 1, device=DEV, generator=g))
            sc = x.abs().amax(-1) / 448.0
            codes[p, :, :live] = (x / sc[..., None]).to(torch.float8_e4m3fn)
            scale[p, :, :live] = sc
        out += [codes, scale]
    return out


def _rope(max_pos, rd=64, theta=1e7):
    inv = 1.0 / theta ** (torch.arange(0, rd, 2, dtype=F32, device=DEV) / rd)
    f = torch.arange(max_pos, dtype=F32, device=DEV)[:, None] * inv[None]
    e = torch.cat([f, f], -1)
    return e.cos().to(BF), e.sin().to(BF)


def _gdn_weights(g, hidden, h, hv):
    c = 2 * h * 128 + hv * 128
    return {"in_ba": _randn(g, 2 * hv, hidden, std=0.02), "conv_w": _randn(g, c, 4, std=0.3),
            "a_log": torch.randn(hv, device=DEV, generator=g), "dt_bias": torch.randn(hv, device=DEV, generator=g),
            "norm_w": _randn(g, 128, std=0.5, mean=1.0)}


# ------------------------------------------------------------------ float64 forms

def _w64(w, lo=0, hi=None):
    """q * s + mn in float64 (rows lo..hi)."""
    q, s, mn = (t[lo:hi] for t in w)
    codes = torch.stack([q & 15, q >> 4], -1).view(q.shape[0], s.shape[1], 128).to(F64)
    return (codes * s.to(F64)[..., None] + mn.to(F64)[..., None]).view(q.shape[0], -1)


def _lin64(x, w):
    return torch.cat([x.to(F64) @ _w64(w, i, i + 16384).T for i in range(0, w[0].shape[0], 16384)], -1)


def _norm64(x, w):
    x = x.to(F64)
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * (1.0 + w.to(F64))


def _silu64(x):
    return x * torch.sigmoid(x)


def _path(parent, t):
    p = [t]
    while parent[p[-1]] >= 0:
        p.append(parent[p[-1]])
    return p[::-1]


def _gdn64(u, n, w, ring, rec0, pos, parent, h, hv):
    """u [M, C + HV V], n [M, hidden], ring [C, R], rec0 [HV, K, V] -> (y [M, HV V], states [M, HV, K, V])."""
    M, qk = u.shape[0], h * 128
    C = 2 * qk + hv * 128
    u = u.to(F64)
    cw, ring = w["conv_w"].to(F64), ring.to(F64)
    ba = n.to(F64) @ w["in_ba"].to(F64).T
    beta = torch.sigmoid(ba[:, :hv])
    decay = torch.exp(-torch.exp(w["a_log"].to(F64)) * torch.nn.functional.softplus(ba[:, hv:] + w["dt_bias"].to(F64)))
    back = [ring[:, (pos + j - 3) % RING] for j in range(3)]
    y, states = [], []
    for t in range(M):
        rows = (back + [u[i, :C] for i in _path(parent, t)])[-4:]
        c = _silu64(sum(r * cw[:, j] for j, r in enumerate(rows)))
        q, k, v = c[:qk].view(h, 128), c[qk:2 * qk].view(h, 128), c[2 * qk:].view(hv, 128)
        q = q * torch.rsqrt(q.square().sum(-1, keepdim=True) + 1e-6) * 128 ** -0.5
        k = k * torch.rsqrt(k.square().sum(-1, keepdim=True) + 1e-6)
        q, k = q.repeat_interleave(hv // h, 0), k.repeat_interleave(hv // h, 0)
        S = (rec0.to(F64) if parent[t] < 0 else states[parent[t]]) * decay[t][:, None, None]
        dv = beta[t][:, None] * (v - (k[:, :, None] * S).sum(1))
        S = S + k[:, :, None] * dv[:, None, :]
        o = (q[:, :, None] * S).sum(1)
        o = o * torch.rsqrt(o.square().mean(-1, keepdim=True) + EPS) * w["norm_w"].to(F64)
        y.append((o * _silu64(u[t, C:].view(hv, 128))).reshape(-1))
        states.append(S)
    return torch.stack(y), torch.stack(states)


def _attn64(u, qw, kw, k, ks, v, vs, pos, parent, hq, hkv):
    """u [M, HQ 2D + 2 HKV D], caches [HKV, maxlen, D] with scales, rows < pos live -> y [M, HQ D]."""
    M, D, G = u.shape[0], 256, hq // hkv
    u = u.to(F64)
    cos, sin = (t.to(F64) for t in _rope(pos + M))

    def roped(x, w):
        x = _norm64(x, w)
        out = []
        for t in range(M):
            p = pos + len(_path(parent, t)) - 1
            a, b, r = x[t, :, :32], x[t, :, 32:64], x[t, :, 64:]
            c, s = cos[p, :32], sin[p, :32]
            out.append(torch.cat([a * c - b * s, b * c + a * s, r], -1))
        return torch.stack(out)

    def stored(x):   # what a cache row holds of [M, HKV, D]
        sc = x.abs().amax(-1, keepdim=True) / 448.0
        return (x / sc).to(F32).to(torch.float8_e4m3fn).to(F64) * sc

    qg = u[:, :hq * 2 * D].view(M, hq, 2, D)
    q, gate = roped(qg[:, :, 0], qw), torch.sigmoid(qg[:, :, 1])
    kn = stored(roped(u[:, hq * 2 * D:hq * 2 * D + hkv * D].reshape(M, hkv, D), kw))
    vn = stored(u[:, hq * 2 * D + hkv * D:].reshape(M, hkv, D))
    sees = torch.zeros(M, M, dtype=torch.bool, device=DEV)
    for t in range(M):
        sees[t, _path(parent, t)] = True
    y = torch.empty(M, hq, D, dtype=F64, device=DEV)
    for j in range(hkv):
        K = torch.cat([k[j, :pos].to(F64) * ks[j, :pos, None].to(F64), kn[:, j]])
        V = torch.cat([v[j, :pos].to(F64) * vs[j, :pos, None].to(F64), vn[:, j]])
        for h in range(j * G, j * G + G):
            s = q[:, h] @ K.T / 16.0
            s[:, pos:] = s[:, pos:].masked_fill(~sees, -math.inf)
            y[:, h] = torch.softmax(s, -1) @ V
    return (y * gate).reshape(M, -1)


# ------------------------------------------------------------------ capture

def _captured(fn):
    """fn's launches as one hipGraph, after a warm call that allocates every workspace."""
    fn()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = fn()
    return g, out


def _qlinear(w, **kw):
    from tokenrush_amd.quant import QLinear
    return QLinear(*w, **kw)


# ------------------------------------------------------------------ kinds

class Proj:
    """A stack of independent N x K projections, QLinear's call at M rows each."""

    @staticmethod
    def make(c, seed):
        g = _gen(seed)
        return [(_weight(g, c["n"], c["k"], c["scale"]), _randn(g, c["m"], c["k"])) for _ in range(c["layers"])]

    @staticmethod
    def prepare(c, seed):
        stack = [(_qlinear(w), x) for w, x in Proj.make(c, seed)]
        return _captured(lambda: [lin(x) for lin, x in stack]) + (stack,)

    @staticmethod
    def exact(c, seed):
        return [_lin64(x, w) for w, x in Proj.make(c, seed)]

    @staticmethod
    def work(c):
        m, n, k = c["m"], c["n"], c["k"]
        return c["layers"] * (n * k // 2 + n * k // 32 + 2 * m * (n + k)), c["layers"] * 2 * m * n * k


class LayerSet:
    """The projections and norms of layers as the step runs them, around given mixer outputs y:
    u = qkv(n), (x, n) = add_rmsnorm(x, o(y) partials), a = silu_mul(gate_up(n)),
    (x, n) = add_rmsnorm(x, down(a) partials)."""

    @staticmethod
    def make(c, seed):
        g = _gen(seed)
        h, m = c["hidden"], c["m"]
        return [{"qkv": _weight(g, c["qkv"], h, c["scale"]), "o": _weight(g, h, c["attn"], c["scale"]),
                 "gate_up": _weight(g, 2 * c["mlp"], h, c["scale"]), "down": _weight(g, h, c["mlp"], c["scale"]),
                 "ln1": _randn(g, h, std=0.1), "ln2": _randn(g, h, std=0.1), "x": _randn(g, m, h), "n": _randn(g, m, h),
                 "y": _randn(g, m, c["attn"])} for _ in range(c["layers"])]

    @staticmethod
    def prepare(c, seed):
        from tokenrush_amd.fused import add_rmsnorm
        layers = LayerSet.make(c, seed)
        for L in layers:
            L.update(qkv=_qlinear(L["qkv"]), o=_qlinear(L["o"], split_k=4),
                     gate_up=_qlinear(L["gate_up"], layout="gate_up"), down=_qlinear(L["down"], split_k=4))

        def step():
            out = []
            for L in layers:
                u = L["qkv"](L["n"])
                x, n = add_rmsnorm(L["x"], L["o"].partials(L["y"]), L["ln1"], EPS)
                a = L["gate_up"].silu_mul(n)
                out += [u, x, n, a, *add_rmsnorm(x, L["down"].partials(a), L["ln2"], EPS)]
            return out
        return _captured(step) + (layers,)

    @staticmethod
    def exact(c, seed):
        out = []
        for L in LayerSet.make(c, seed):
            u = _lin64(L["n"], L["qkv"])
            x = L["x"].to(F64) + _lin64(L["y"], L["o"])
            n = _norm64(x, L["ln1"])
            gu = _lin64(n, L["gate_up"])
            a = _silu64(gu[:, :c["mlp"]]) * gu[:, c["mlp"]:]
            x2 = x + _lin64(a, L["down"])
            out += [u, x, n, a, x2, _norm64(x2, L["ln2"])]
        return out

    @staticmethod
    def work(c):
        h, m = c["hidden"], c["m"]
        shapes = [(c["qkv"], h), (h, c["attn"]), (2 * c["mlp"], h), (h, c["mlp"])]
        nk = sum(n * k for n, k in shapes)
        return (c["layers"] * (nk // 2 + nk // 32 + 2 * m * (c["qkv"] + c["attn"] + c["mlp"] + 6 * h)),
                c["layers"] * 2 * m * nk)


class Mlp:
    """down(silu_mul(gate_up(x))) of a prompt: more rows than a verify step has, called eagerly."""

    @staticmethod
    def make(c, seed):
        g = _gen(seed)
        return _weight(g, 2 * c["mlp"], c["hidden"]), _weight(g, c["hidden"], c["mlp"]), _randn(g, c["t"], c["hidden"])

    @staticmethod
    def prepare(c, seed):
        gate_up, down, x = Mlp.make(c, seed)
        return _qlinear(gate_up, layout="gate_up"), _qlinear(down, split_k=4), x

    @staticmethod
    def exact(c, seed):
        gate_up, down, x = Mlp.make(c, seed)
        gu = _lin64(x, gate_up)
        a = _silu64(gu[:, :c["mlp"]]) * gu[:, c["mlp"]:]
        return [a, _lin64(a, down)]

    @staticmethod
    def work(c):
        h, f, t = c["hidden"], c["mlp"], c["t"]
        return 3 * h * f // 2 + 3 * h * f // 32 + 2 * t * (2 * h + f), 6 * t * h * f


class Gdn:
    """gdn_step_fused of a few independent layers: a chain of M tokens or an M-node draft tree. The
    committed state sits in a slot of its own, so every pass starts from the same state."""

    @staticmethod
    def make(c, seed):
        g = _gen(seed)
        C = 2 * c["h"] * 128 + c["hv"] * 128
        layers = [dict(_gdn_weights(g, c["hidden"], c["h"], c["hv"]), u=_randn(g, c["m"], C + c["hv"] * 128),
                       n=_randn(g, c["m"], c["hidden"]), ring=_randn(g, C, RING)) for _ in range(c["layers"])]
        rec = torch.randn(c["m"] + 1, c["layers"], c["hv"], 128, 128, device=DEV, generator=g) * 0.05
        return layers, rec, _parents(c, seed)

    @staticmethod
    def prepare(c, seed):
        from tokenrush_amd.gdn import GDNConfig, gdn_step_fused
        layers, rec, parent = Gdn.make(c, seed)
        cfg = GDNConfig(c["hidden"], c["h"], c["hv"], 128, 128)
        pos = torch.tensor([c["pos"]], device=DEV)
        slot = torch.tensor([c["m"]], device=DEV)
        par = torch.tensor(parent, dtype=torch.int32, device=DEV) if c["tree"] else None
        for L in layers:
            L["A"] = -torch.exp(L["a_log"])
            L["node_in"] = torch.zeros(c["m"], cfg.conv_dim, dtype=BF, device=DEV) if c["tree"] else None

        def step():
            return [gdn_step_fused(L["u"], L["n"], L["in_ba"], L["ring"], L["conv_w"], L["A"], L["dt_bias"], rec[:, i],
                                   slot, L["norm_w"], pos, cfg, EPS, parent=par, node_in=L["node_in"])
                    for i, L in enumerate(layers)]
        g, ys = _captured(step)
        out = [[y, rec[:c["m"], i], L["node_in"] if c["tree"] else L["ring"]]
               for i, (y, L) in enumerate(zip(ys, layers))]
        return g, out, (layers, pos, slot, par)

    @staticmethod
    def exact(c, seed):
        layers, rec, parent = Gdn.make(c, seed)
        return [list(_gdn64(L["u"], L["n"], L, L["ring"], rec[c["m"], i], c["pos"], parent, c["h"], c["hv"])) + [None]
                for i, L in enumerate(layers)]

    @staticmethod
    def work(c):
        m, h, hv = c["m"], c["h"], c["hv"]
        C = 2 * h * 128 + hv * 128
        per = (m + 1) * hv * 65536 + 2 * m * (C + 2 * hv * 128 + c["hidden"]) + 4 * hv * c["hidden"] + 2 * C * (7 + m)
        return c["layers"] * per, c["layers"] * m * hv * 128 * 128 * 8


class Attn:
    """attn_prep then attn_decode_fused of a few independent layers over `ctx` live tokens: M chain
    tokens or an M-node draft tree."""

    @staticmethod
    def make(c, seed):
        g = _gen(seed)
        hq, hkv = c["hq"], c["hkv"]
        layers = [{"u": _randn(g, c["m"], hq * 512 + hkv * 512), "qw": _randn(g, 256, std=0.5),
                   "kw": _randn(g, 256, std=0.5)} for _ in range(c["layers"])]
        return layers, _cache(g, c["layers"], hkv, c["ctx"] + 64, c["ctx"]), _parents(c, seed)

    @staticmethod
    def prepare(c, seed):
        from tokenrush_amd.attn import AttnConfig, attn_decode_fused, attn_prep
        layers, (k, ks, v, vs), parent = Attn.make(c, seed)
        cfg = AttnConfig(c["hq"], c["hkv"], 256, 64, 1e7, EPS)
        cos, sin = _rope(c["ctx"] + 64)
        pos = torch.tensor([c["ctx"]], device=DEV)
        par = torch.tensor(parent, dtype=torch.int32, device=DEV) if c["tree"] else None

        def step():
            out = []
            for i, L in enumerate(layers):
                q = attn_prep(L["u"], L["qw"], L["kw"], cos, sin, pos, k[i], v[i], cfg, ks[i], vs[i], parent=par)
                out.append(attn_decode_fused(q, L["u"], k[i], v[i], pos, cfg, ks[i], vs[i], parent=par))
            return out
        g, ys = _captured(step)
        new = slice(c["ctx"], c["ctx"] + c["m"])
        out = [ys, k[:, :, new].view(torch.uint8), v[:, :, new].view(torch.uint8), ks[:, :, new], vs[:, :, new]]
        return g, out, (layers, cos, sin, pos, par)

    @staticmethod
    def exact(c, seed):
        layers, (k, ks, v, vs), parent = Attn.make(c, seed)
        ys = [_attn64(L["u"], L["qw"], L["kw"], k[i], ks[i], v[i], vs[i], c["ctx"], parent, c["hq"], c["hkv"])
              for i, L in enumerate(layers)]
        return [ys, None, None, None, None]

    @staticmethod
    def work(c):
        m, hq, hkv, L = c["m"], c["hq"], c["hkv"], c["ctx"] + c["m"]
        return (c["layers"] * (L * hkv * 520 + 2 * m * (hq + hkv) * 512 + 2 * m * hq * 256),
                c["layers"] * 4 * m * hq * L * 256)


class Accept:
    """One verify accept: peaked logits as a model's are, drafts that match a prefix of the rows' peaks."""

    @staticmethod
    def make(c, seed):
        g = _gen(seed)
        m, v = c["m"], c["v"]
        lg = torch.randn(m, v, device=DEV, generator=g) * 2
        peak = torch.randint(0, v, (m,), device=DEV, generator=g)
        lg[torch.arange(m, device=DEV), peak] += 14.0
        toks = torch.randint(0, v, (m,), device=DEV, generator=g)
        parent = _tree(m, seed) if c["rule"] == "tree" else list(range(-1, m - 1))
        for i in range(1, m):                # the first nodes hold what their parent's row predicts
            if i <= m // 2:
                toks[i] = peak[parent[i]]
        u = torch.rand(m, device=DEV, generator=g)
        q = None
        if c["rule"] == "residual":
            q = torch.softmax(lg[:-1] + torch.randn(m - 1, v, device=DEV, generator=g), -1)
        return lg.to(BF), toks, parent, u, q

    @staticmethod
    def prepare(c, seed):
        from tokenrush_amd.accept import AcceptState, accept_greedy, accept_residual, accept_sampled, accept_tree
        from tokenrush_amd.sample import SamplingParams
        lg, toks, parent, u, q = Accept.make(c, seed)
        st = AcceptState(c["m"], DEV)
        params = SamplingParams(DEV)
        params.set(temperature=0.8, top_p=0.95, top_k=40)
        par = torch.tensor(parent, dtype=torch.int32, device=DEV)
        call = {"greedy": lambda: accept_greedy(lg, toks, st), "tree": lambda: accept_tree(lg, toks, par, st),
                "sampled": lambda: accept_sampled(lg, toks, params, st, u),
                "residual": lambda: accept_residual(lg, q, toks, u, st)}[c["rule"]]
        g, _ = _captured(call)
        return g, [st.n_accepted, st.tok, st.slot, st.tokens, st.pos], (lg, toks, u, q, par, params, st)

    @staticmethod
    def exact(c, seed):
        return None      # token ids and counts only

    @staticmethod
    def work(c):
        m, v = c["m"], c["v"]
        return 2 * m * v + (4 * v if c["rule"] == "residual" else 0) + 64 * m, 4 * m * v


class Load:
    """One matrix into the kernel layout (QLinear's construction), back to the engine packing (as a
    checkpoint is saved) and to a dense matrix."""

    @staticmethod
    def make(c, seed):
        return _weight(_gen(seed), c["n"], c["k"])

    @staticmethod
    def prepare(c, seed):
        return c, Load.make(c, seed)

    @staticmethod
    def exact(c, seed):
        return [None, None, None, _w64(Load.make(c, seed))]

    @staticmethod
    def work(c):
        packed = c["n"] * c["k"] // 2 + c["n"] * c["k"] // 32
        return 5 * packed + 2 * c["n"] * c["k"], c["n"] * c["k"] * 2


class Step:
    """VerifyModel over one period of the hybrid: a greedy chain step from token ids (verify) or a
    draft-tree step (step_tree). Drafts are random tokens, so the root alone is accepted."""

    @staticmethod
    def cfg(c):
        from tokenrush_amd.step import StepConfig
        return StepConfig(n_layers=4, hidden=c["hidden"], mlp=c["mlp"], vocab=c["vocab"], live=c["ctx"], headroom=64,
                          tree_nodes=32 if c["tree"] else 0)

    @staticmethod
    def make(c, seed):
        g = _gen(seed)
        hid, f, t = c["hidden"], c["mlp"], {}

        def put(name, n, k):
            for suffix, v in zip((".qweight", ".scale", ".mn"), _weight(g, n, k)):
                t[name + suffix] = v
        for li in range(4):
            p = "layers.%d." % li
            if li == 3:
                p += "self_attn."
                put(p + "q_proj.weight", 24 * 512, hid)
                put(p + "k_proj.weight", 1024, hid)
                put(p + "v_proj.weight", 1024, hid)
                put(p + "o_proj.weight", hid, 6144)
                t[p + "q_norm.weight"], t[p + "k_norm.weight"] = _randn(g, 256, std=0.5), _randn(g, 256, std=0.5)
            else:
                p += "linear_attn."
                w = _gdn_weights(g, hid, 16, 48)
                put(p + "in_proj_qkv.weight", 10240, hid)
                put(p + "in_proj_z.weight", 6144, hid)
                put(p + "out_proj.weight", hid, 6144)
                t.update({p + "in_proj_b.weight": w["in_ba"][:48], p + "in_proj_a.weight": w["in_ba"][48:],
                          p + "conv1d.weight": w["conv_w"].unsqueeze(1), p + "A_log": w["a_log"],
                          p + "dt_bias": w["dt_bias"], p + "norm.weight": w["norm_w"]})
            p = "layers.%d." % li
            put(p + "mlp.gate_proj.weight", f, hid)
            put(p + "mlp.up_proj.weight", f, hid)
            put(p + "mlp.down_proj.weight", hid, f)
            t[p + "input_layernorm.weight"] = _randn(g, hid, std=0.1)
            t[p + "post_attention_layernorm.weight"] = _randn(g, hid, std=0.1)
        put("lm_head.weight", c["vocab"], hid)
        t["norm.weight"] = _randn(g, hid, std=0.1)
        t["embed_tokens.weight"] = _randn(g, c["vocab"], hid)
        slots = 32 if c["tree"] else 8
        return {"tensors": t, "ring": _randn(g, 3, 10240, RING),
                "rec": torch.randn(slots, 3, 48, 128, 128, device=DEV, generator=g) * 0.05,
                "cache": _cache(g, 1, 4, c["ctx"] + 64, c["ctx"]),
                "toks": torch.randint(0, c["vocab"], (c["m"],), device=DEV, generator=g),
                "parent": _parents(c, seed)}

    @staticmethod
    def prepare(c, seed):
        from tokenrush_amd.accept import AcceptState
        from tokenrush_amd.step import VerifyModel
        r = Step.make(c, seed)
        model = VerifyModel(Step.cfg(c), device=DEV, seed=0, tensors=r["tensors"])
        S = model.state

        def reset():
            S.ring.copy_(r["ring"])
            S.rec.copy_(r["rec"])
            for a, b in zip((S.k, S.k_scale, S.v, S.v_scale), r["cache"]):
                a.copy_(b)
            S.pos.fill_(c["ctx"])
            S.slot.zero_()
        st = AcceptState(c["m"], DEV, pos=S.pos)
        st.slot = S.slot
        toks, par = r["toks"], torch.tensor(r["parent"], dtype=torch.int32, device=DEV)
        x0 = model.embed[toks].contiguous()

        def step():
            S.pos.fill_(c["ctx"])      # every pass at the same position, from the state the last one left
            return model.step_tree(x0, toks, par, st) if c["tree"] else model.verify(toks, st)
        reset()
        g, logits = _captured(step)
        reset()
        return g, [logits, S.rec[:c["m"]], S.pos, st.n_accepted], (model, r["toks"], x0, par, st)

    @staticmethod
    def exact(c, seed):
        r = Step.make(c, seed)
        t, parent = r["tensors"], r["parent"]
        w = lambda *names: tuple(torch.cat([t[n + s] for n in names]) for s in (".qweight", ".scale", ".mn"))
        x, states = t["embed_tokens.weight"][r["toks"]].to(F64), []
        for li in range(4):
            p = "layers.%d." % li
            n = _norm64(x, t[p + "input_layernorm.weight"])
            if li == 3:
                a = p + "self_attn."
                u = _lin64(n, w(a + "q_proj.weight", a + "k_proj.weight", a + "v_proj.weight"))
                k, ks, v, vs = (z[0] for z in r["cache"])
                y = _attn64(u, t[a + "q_norm.weight"], t[a + "k_norm.weight"], k, ks, v, vs, c["ctx"], parent, 24, 4)
                out = a + "o_proj.weight"
            else:
                a = p + "linear_attn."
                u = _lin64(n, w(a + "in_proj_qkv.weight", a + "in_proj_z.weight"))
                gw = {"in_ba": torch.cat([t[a + "in_proj_b.weight"], t[a + "in_proj_a.weight"]]),
                      "conv_w": t[a + "conv1d.weight"].squeeze(1), "a_log": t[a + "A_log"], "dt_bias": t[a + "dt_bias"],
                      "norm_w": t[a + "norm.weight"]}
                y, s = _gdn64(u, n, gw, r["ring"][li], r["rec"][0, li], c["ctx"], parent, 16, 48)
                states.append(s)
                out = a + "out_proj.weight"
            x = x + _lin64(y, w(out))
            n = _norm64(x, t[p + "post_attention_layernorm.weight"])
            h = _silu64(_lin64(n, w(p + "mlp.gate_proj.weight"))) * _lin64(n, w(p + "mlp.up_proj.weight"))
            x = x + _lin64(h, w(p + "mlp.down_proj.weight"))
        return [_lin64(_norm64(x, t["norm.weight"]), w("lm_head.weight")), torch.stack(states, 1), None, None]

    @staticmethod
    def work(c):
        h, f, m = c["hidden"], c["mlp"], c["m"]
        nk = 3 * (16384 * h + 6144 * h) + 14336 * h + 6144 * h + 4 * 3 * h * f + c["vocab"] * h
        mix = 3 * (m + 1) * 48 * 65536 + (c["ctx"] + m) * 4 * 520
        return nk // 2 + nk // 32 + mix + 2 * m * c["vocab"], 2 * m * nk


KINDS = {"proj": Proj, "layer": LayerSet, "mlp": Mlp, "gdn": Gdn, "attn": Attn, "accept": Accept, "load": Load,
         "step": Step}


def prepare(case, seed):
    return case["kind"], KINDS[case["kind"]].prepare(case, seed)


def run(state):
    kind, s = state
    if kind == "mlp":
        gate_up, down, x = s
        a = gate_up.silu_mul(x)
        return [a, down(a)]
    if kind == "load":
        c, w = s
        lin = _qlinear(w, layout=c["layout"])
        return [*lin.nibbles(), lin.dequantize()]
    s[0].replay()
    return s[1]


def exact(case, seed):
    return KINDS[case["kind"]].exact(case, seed)


def work(case):
    b, f = KINDS[case["kind"]].work(case)
    return {"bytes": b, "flops": f}


def tolerance(case):
    """Four times the error against float64 that the path's data types show, see exact()."""
    kind = case["kind"]
    if kind in ("accept", "load"):
        return "exact"                      # token ids and counts; codes, parameters and their two-rounding product
    if kind == "proj":
        return {"rel": 7e-3, "max": 0.03}   # one bf16 rounding of a 32-bit sum (0.0017 seen)
    if kind in ("layer", "mlp", "step"):
        return {"rel": 0.02, "max": 0.2}    # bf16 between the layer's products (0.006 seen)
    if kind == "gdn":
        return {"rel": 0.02, "max": 0.2}    # bf16 conv outputs, gates and norm (0.005 seen)
    return {"rel": 0.03, "max": 0.3, "differ": 0.01}   # bf16 keys and probabilities (0.008 seen); fp8 codes at ties
