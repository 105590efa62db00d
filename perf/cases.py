"""The work that users of soinfer give it, as cases that can be timed.

Each case is one call, or one whole generation, through the public entry points (soinfer.ops, soinfer.quant,
soinfer.runtime): the single operators at the sizes of the decoder shapes this repository runs (Qwen3 0.6B to 14B
linears), one DIP MLP, and the decode engine from prompt to new tokens.

Weights are W ~ N(0, 0.02) quantized symmetrically (INT4 / INT8, one fp32 scale per group), activations N(0, 1) in
binary16. The engine's decoder ties its LM head to the embedding, as the small Qwen3 checkpoints do, so greedy
tokens have the margin of a real model's and do not hang on the last bit of a logit.
"""
from __future__ import annotations

import math
import sys
from pathlib import Path

import numpy as np
import torch

_PKG = str(Path(__file__).resolve().parent.parent / "sparse-offload-infer_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

GS = 128  # quantization group of every linear
QWEN3_1P7B = dict(H=2048, I=6144, NQ=16, NKV=8, hd=128)


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------

def listed():
    return [
        # one INT4 linear, the smallest of the decoder (k_proj / v_proj): a call's fixed cost
        dict(name="gemv_int4_kv", kind="gemv", bits=4, N=1024, K=2048, gs=GS),
        # one INT8 linear with group scales, down_proj
        dict(name="gemv_int8_down", kind="gemv", bits=8, N=2048, K=6144, gs=GS),
        # every linear of the 28-layer decoder as one grouped launch (the repository's headline benchmark)
        dict(name="gemv_group_28l", kind="group", layers=28, H=2048, I=6144, NQ=16, NKV=8, hd=128),
        # the channel selection of Dynamic Input Pruning at the 1.7B width
        dict(name="topk_6144", kind="topk", n=6144, k=3072),
        # one DIP MLP over resident weights
        dict(name="dip_mlp_half", kind="dip_mlp", H=2048, I=6144, k=3072),
        # one cache-aware DIP MLP: 20% of the channels resident, the misses gathered from pinned host memory
        dict(name="cached_dip_mlp_20", kind="cached_dip_mlp", H=2048, I=6144, k=3072, hot=0.2),
        # decode attention late in a 2048-token context
        dict(name="attention_1999", kind="attention", NQ=16, NKV=8, hd=128, L=1999, max_seq=2048),
        # loading: one fp32 checkpoint matrix to packed INT4 (up_proj)
        dict(name="quantize_up", kind="quantize", N=6144, K=2048, gs=GS),
        # a prompt to its first new token, dense, the whole 1.7B shape
        dict(name="prompt_dense_256", kind="generate", mode="dense", layers=28, vocab=151936, P=256, n=1, k=0,
             hot=0.0, offload=False, int4_head=False, **QWEN3_1P7B),
        # a short question and a longer answer, dense, the whole 1.7B shape
        dict(name="generate_dense_8_32", kind="generate", mode="dense", layers=28, vocab=151936, P=8, n=32, k=0,
             hot=0.0, offload=False, int4_head=False, **QWEN3_1P7B),
        # a 64-token prompt and 16 new tokens with DIP at half the channels
        dict(name="generate_dip_64_16", kind="generate", mode="dip", layers=28, vocab=151936, P=64, n=16, k=3072,
             hot=0.0, offload=False, int4_head=False, **QWEN3_1P7B),
        # weights kept in host memory and streamed (8 of the layers), a prompt and a few tokens
        dict(name="offload_dense_48_4", kind="generate", mode="dense", layers=8, vocab=151936, P=48, n=4, k=0,
             hot=0.0, offload=True, int4_head=False, **QWEN3_1P7B),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng, lo, hi):
    """A width of a real layer (a multiple of 128) more often than not, else any size."""
    n = _log_int(rng, lo, hi)
    return max(128, n // 128 * 128) if rng.random() < 0.7 else n


def draw(rng):
    kind = rng.choice(["gemv", "gemv", "group", "topk", "dip_mlp", "cached_dip_mlp", "attention", "quantize",
                       "generate", "generate", "generate", "generate"])
    if kind == "gemv":
        while True:
            N, K = _size(rng, 256, 17408), _size(rng, 256, 17408)
            if N * K <= 17408 * 5120:
                return dict(kind=kind, bits=rng.choice([4, 4, 8]), N=N, K=K, gs=rng.choice([64, 128, 128]))
    if kind == "group":
        return dict(kind=kind, layers=rng.randint(1, 12), H=128 * rng.randint(4, 20), I=128 * rng.randint(8, 60),
                    NQ=rng.choice([8, 16, 32]), NKV=8, hd=rng.choice([64, 128]))
    if kind == "topk":
        n = _log_int(rng, 256, 27648)
        return dict(kind=kind, n=n, k=max(1, int(n * rng.uniform(0.1, 0.6))))
    if kind in ("dip_mlp", "cached_dip_mlp"):
        I = 128 * _log_int(rng, 6, 100)
        c = dict(kind=kind, H=128 * _log_int(rng, 4, 32), I=I, k=max(1, int(I * rng.uniform(0.1, 0.6))))
        if kind == "cached_dip_mlp":
            c["hot"] = round(rng.uniform(0.0, 0.8), 3)
        return c
    if kind == "attention":
        kv, L = rng.choice([2, 4, 8]), _log_int(rng, 1, 16384)
        return dict(kind=kind, NQ=kv * rng.choice([1, 2, 4]), NKV=kv, hd=rng.choice([64, 128]), L=L,
                    max_seq=L + rng.randint(0, 512))
    if kind == "quantize":
        return dict(kind=kind, N=_size(rng, 256, 12288), K=_size(rng, 256, 12288), gs=rng.choice([64, 128, 128]))
    kv, I = rng.choice([1, 2, 4, 8]), 128 * _log_int(rng, 4, 48)
    mode = rng.choice(["dense", "dense", "dip", "cached_dip"])
    return dict(kind="generate", mode=mode, layers=rng.randint(1, 6), H=128 * _log_int(rng, 2, 24), I=I,
                NQ=kv * rng.choice([1, 2, 4]), NKV=kv, hd=rng.choice([64, 128]), vocab=_log_int(rng, 2000, 100000),
                P=_log_int(rng, 1, 400), n=_log_int(rng, 1, 24),
                k=0 if mode == "dense" else max(1, int(I * rng.uniform(0.2, 0.6))),
                hot=round(rng.uniform(0.1, 0.6), 3) if mode == "cached_dip" else 0.0,
                offload=mode != "dip" and rng.random() < 0.3, int4_head=rng.random() < 0.3)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

_DEV = "cuda"
_ORDER = (0, 2, 4, 6, 1, 3, 5, 7)  # nibble i of a word holds value _ORDER[i] of its eight


def _gen(seed):
    return torch.Generator(device=_DEV).manual_seed(int(seed))


def _codes(g, N, K, gs, bits=4):
    """(q int8 [N, K], scale fp32 [N, ceil(K/gs)]) of W ~ N(0, 0.02)."""
    qmax = (1 << (bits - 1)) - 1
    G = -(-K // gs)
    w = torch.zeros(N, G * gs, device=_DEV)
    w[:, :K] = torch.randn(N, K, generator=g, device=_DEV) * 0.02
    w = w.view(N, G, gs)
    s = w.abs().amax(-1).div_(qmax).clamp_(min=1e-30)
    q = (w / s[..., None]).round_().clamp_(-qmax, qmax).to(torch.int8).view(N, G * gs)[:, :K]
    return q.contiguous(), s.contiguous()


def _packed(q):
    """AWQ-order packed rows, uint8 [N, ceil(K/8)*4]."""
    N, K = q.shape
    words = -(-K // 8)
    v = torch.zeros(N, words * 8, dtype=torch.int32, device=q.device)
    v[:, :K] = q
    v = (v & 15).view(N, words, 8)
    out = torch.zeros(N, words, dtype=torch.int32, device=q.device)
    for i, j in enumerate(_ORDER):
        out |= v[..., j] << (4 * i)
    return out.view(torch.uint8).view(N, words * 4).contiguous()


def _deq(q, s, gs):
    """The quantized matrix in 64 bits."""
    N, K = q.shape
    return q.double() * s.double().repeat_interleave(gs, 1)[:, :K]


def _x(g, n):
    return torch.randn(n, generator=g, device=_DEV).half()


def _group_shapes(c):
    qd, kvd = c["NQ"] * c["hd"], c["NKV"] * c["hd"]
    return [(qd, c["H"]), (kvd, c["H"]), (kvd, c["H"]), (c["H"], qd), (c["I"], c["H"]), (c["I"], c["H"]),
            (c["H"], c["I"])] * c["layers"]


def _group_inputs(c, seed):
    g = _gen(seed)
    return [(*_codes(g, N, K, GS), _x(g, K), K) for N, K in _group_shapes(c)]


def _mlp_inputs(c, seed):
    g = _gen(seed)
    return dict(gate=_codes(g, c["I"], c["H"], GS), up=_codes(g, c["I"], c["H"], GS),
                down=_codes(g, c["I"], c["H"], GS), x=_x(g, c["H"]),
                hot=torch.randperm(c["I"], generator=g, device=_DEV)[:int(c.get("hot", 0.0) * c["I"])].sort().values)


def _linears(c):
    qkv = (c["NQ"] + 2 * c["NKV"]) * c["hd"]
    return [("qkv", qkv, c["H"]), ("o", c["H"], c["NQ"] * c["hd"]), ("gu", 2 * c["I"], c["H"])]


def _decoder_inputs(c, seed):
    """Codes, norms, embedding and prompt of a decoder; down_proj is quantized as [H, I] for the dense path and as
    its transpose for DIP."""
    g = _gen(seed)

    def norm(n):
        return (1.0 + 0.1 * torch.randn(n, generator=g, device=_DEV)).half()

    layers = []
    for _ in range(c["layers"]):
        L = {name: _codes(g, N, K, GS) for name, N, K in _linears(c)}
        L["down"] = _codes(g, c["H"], c["I"], GS)
        L["down_T"] = _codes(g, c["I"], c["H"], GS) if c["mode"] != "dense" else None
        L["norms"] = (norm(c["H"]), norm(c["H"]), norm(c["hd"]), norm(c["hd"]))
        layers.append(L)
    embed = torch.empty(c["vocab"], c["H"], dtype=torch.float16, device=_DEV).normal_(generator=g)
    hot = [torch.randperm(c["I"], generator=g, device=_DEV)[:int(c["hot"] * c["I"])].sort().values.tolist()
           for _ in range(c["layers"])] if c["mode"] == "cached_dip" else None
    prompt = torch.randint(0, c["vocab"], (c["P"],), generator=g, device=_DEV).tolist()
    return dict(layers=layers, embed=embed, final_norm=norm(c["H"]), prompt=prompt, hot=hot)


def prepare(case, seed):
    c, kind = case, case["kind"]
    if kind == "gemv":
        from soinfer import ops

        g = _gen(seed)
        q, s = _codes(g, c["N"], c["K"], c["gs"], c["bits"])
        return dict(c=c, fn=ops.gemv_w4a16_group_lop3 if c["bits"] == 4 else ops.gemv_w8a16,
                    W=_packed(q) if c["bits"] == 4 else q, s=s, x=_x(g, c["K"]))
    if kind == "group":
        from soinfer import ops

        probs = [(_packed(q), s, x, K) for q, s, x, K in _group_inputs(c, seed)]
        y = torch.empty(sum(p[0].shape[0] for p in probs), dtype=torch.float16, device=_DEV)
        ys = list(y.split([p[0].shape[0] for p in probs]))
        return dict(c=c, group=ops.GemvGroup(probs, GS, ys=ys), y=y)
    if kind == "topk":
        from soinfer import ops

        return dict(c=c, fn=ops.topk_threshold_select, g=_x(_gen(seed), c["n"]).float().abs())
    if kind in ("dip_mlp", "cached_dip_mlp"):
        from soinfer.offload.hot_cache import HotCache
        from soinfer.runtime import dip

        t = _mlp_inputs(c, seed)
        w = dip.DipMLPWeights(_packed(t["gate"][0]), t["gate"][1], _packed(t["up"][0]), t["up"][1],
                              _packed(t["down"][0]), t["down"][1], c["H"], GS)
        st = dict(c=c, dip=dip, w=w, x=t["x"])
        if kind == "cached_dip_mlp":
            st["cache"] = HotCache.build(w.up_Wq, w.up_scale, w.down_T_Wq, w.down_T_scale, t["hot"].tolist())
            st["host"] = [torch.empty(m.shape, dtype=torch.uint8, pin_memory=True).copy_(m)
                          for m in (w.up_Wq, w.down_T_Wq)]
            st["staging"] = torch.empty(c["k"], w.up_Wq.shape[1], dtype=torch.uint8, pin_memory=True)
        return st
    if kind == "attention":
        from soinfer import ops

        g = _gen(seed)
        return dict(c=c, fn=ops.decode_attention, q=_x(g, c["NQ"] * c["hd"]).view(c["NQ"], c["hd"]),
                    k=_x(g, c["NKV"] * c["max_seq"] * c["hd"]).view(c["NKV"], c["max_seq"], c["hd"]),
                    v=_x(g, c["NKV"] * c["max_seq"] * c["hd"]).view(c["NKV"], c["max_seq"], c["hd"]))
    if kind == "quantize":
        from soinfer.quant import formats, pack

        return dict(c=c, formats=formats, pack=pack, cfg=formats.QuantConfig(4, "group", c["gs"]),
                    W=torch.randn(c["N"], c["K"], generator=_gen(seed), device=_DEV) * 0.02)
    from soinfer.runtime import decoder as D

    t = _decoder_inputs(c, seed)
    cfg = D.DecoderConfig(hidden=c["H"], layers=c["layers"], q_heads=c["NQ"], kv_heads=c["NKV"], head_dim=c["hd"],
                          intermediate=c["I"], vocab=c["vocab"], group_size=GS, max_seq=2048)
    layers = []
    for L in t["layers"]:
        m = []
        for name in ("qkv", "o", "gu", "down", "down_T"):
            q, s = L[name] if L[name] is not None else L["gu"]  # the dense engine never reads down^T
            m += [_packed(q), s] if L[name] is not None else [m[4], m[5]]
        layers.append(D.LayerWeights(*L["norms"], *m))
    w = D.DecoderWeights(cfg, t["embed"], t["embed"], t["final_norm"], layers)
    eng = D.DecodeEngine(w, c["mode"], dip_k=c["k"] or None, hot_channels=t["hot"], max_new_tokens=c["n"],
                         offload=c["offload"], int4_head=c["int4_head"])
    eng.capture()
    return dict(c=c, eng=eng, prompt=t["prompt"])


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------

def run(state):
    c, kind = state["c"], state["c"]["kind"]
    if kind == "gemv":
        if c["bits"] == 4:
            return state["fn"](state["W"], state["s"], state["x"], c["K"], c["gs"])
        return state["fn"](state["W"], state["s"], state["x"], c["gs"])
    if kind == "group":
        state["group"].run()
        return state["y"]
    if kind == "topk":
        return state["fn"](state["g"], c["k"])
    if kind == "dip_mlp":
        y, idx = state["dip"].dip_mlp(state["w"], state["x"], c["k"])
        return dict(y=y, idx=idx)
    if kind == "cached_dip_mlp":
        y, idx, misses = state["dip"].cached_dip_mlp(state["w"], state["cache"], state["x"], c["k"], *state["host"],
                                                     state["staging"])
        return dict(y=y, idx=idx, misses=misses)
    if kind == "attention":
        return state["fn"](state["q"], state["k"], state["v"], c["L"])
    if kind == "quantize":
        qt = state["formats"].quantize(state["W"], state["cfg"])
        return dict(packed=state["pack"].pack_int4(qt.qweight)[0], scale=qt.scale)
    eng = state["eng"]
    tokens = eng.generate(state["prompt"], c["n"])
    return dict(tokens=np.array(tokens), logits=eng.logits)


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------

def _int4_bytes(N, K, gs=GS):
    return N * -(-K // 8) * 4 + N * -(-K // gs) * 4


def work(case):
    c, kind = case, case["kind"]
    if kind == "gemv":
        N, K = c["N"], c["K"]
        w = _int4_bytes(N, K, c["gs"]) if c["bits"] == 4 else N * K + N * -(-K // c["gs"]) * 4
        return dict(bytes=w + 2 * K + 2 * N, flops=2 * N * K)
    if kind == "group":
        sh = _group_shapes(c)
        return dict(bytes=sum(_int4_bytes(N, K) + 2 * K + 2 * N for N, K in sh), flops=sum(2 * N * K for N, K in sh))
    if kind == "topk":
        return dict(bytes=4 * c["n"] + 4 * c["k"], flops=0)
    if kind in ("dip_mlp", "cached_dip_mlp"):
        row = _int4_bytes(1, c["H"])
        return dict(bytes=(c["I"] + 2 * c["k"]) * row + 4 * c["H"] + 4 * c["k"],
                    flops=2 * c["H"] * (c["I"] + 2 * c["k"]))
    if kind == "attention":
        return dict(bytes=4 * c["NKV"] * c["L"] * c["hd"] + 4 * c["NQ"] * c["hd"], flops=4 * c["NQ"] * c["L"] * c["hd"])
    if kind == "quantize":
        return dict(bytes=4 * c["N"] * c["K"] + _int4_bytes(c["N"], c["K"], c["gs"]), flops=0)
    # weights once for the whole prompt (every prompt token's layers are known at once) and once per new token
    # (the last new token's layers run too, for the next call); the head once per new token
    H, I, T = c["H"], c["I"], c["P"] + c["n"]
    attn = sum(_int4_bytes(N, K) for name, N, K in _linears(c) if name != "gu")
    dense_mlp = _int4_bytes(2 * I, H) + _int4_bytes(H, I)
    row = _int4_bytes(1, H)
    mlp_new = dense_mlp if c["mode"] == "dense" else (I + 2 * c["k"]) * row
    mlp_prompt = dense_mlp if c["mode"] == "dense" else min(3 * I, I + 2 * c["k"] * c["P"]) * row
    head = _int4_bytes(c["vocab"], H) if c["int4_head"] else 2 * c["vocab"] * H
    kv = 4 * c["NKV"] * c["hd"]
    by = c["layers"] * (attn + mlp_prompt + c["n"] * (attn + mlp_new) + kv * (T + sum(range(c["P"], T)))) + c["n"] * head
    macs = sum(N * K for name, N, K in _linears(c) if name != "gu")
    macs += 3 * H * I if c["mode"] == "dense" else H * (I + 2 * c["k"])
    fl = 2 * T * c["layers"] * macs + 2 * c["n"] * c["vocab"] * H + 2 * c["layers"] * c["NQ"] * c["hd"] * T * T
    return dict(bytes=by, flops=fl)


def tolerance(case):
    """What the data types give. A GEMV or attention output is one binary16 rounding of a binary32 sum (2^-11 of the
    value at most, 2e-4 rms); a DIP output adds the rounding of its h; a whole decoder rounds every layer's result to
    binary16 and carries it through the layers that follow (a dense one: 3e-3 of the logits from the 64-bit result)."""
    kind = case["kind"]
    if kind in ("topk", "quantize"):
        return "exact"
    if kind in ("gemv", "group", "attention"):
        return {"rel": 1e-3}
    if kind in ("dip_mlp", "cached_dip_mlp"):
        return {"rel": 2e-3}
    return {"rel": 2e-2, "max": 0.2}


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------

def _select(g, k):
    """The selection rule over binary32 |gate| [T, n]: 24 bisection steps for the threshold between 0 and the
    maximum, then the first k channels at or above it, as a mask [T, n]."""
    lo = torch.zeros(g.shape[0], 1, device=g.device)
    hi = g.amax(1, keepdim=True) + 1e-3
    for _ in range(24):
        mid = 0.5 * (lo + hi)
        enough = (g >= mid).sum(1, keepdim=True) >= k
        lo, hi = torch.where(enough, mid, lo), torch.where(enough, hi, mid)
    m = g >= lo
    return m & (m.cumsum(1) <= k)


def _silu_mul(g, u):
    return g / (1 + torch.exp(-g)) * u


def _exact_mlp(c, seed):
    t = _mlp_inputs(c, seed)
    x = t["x"].double()
    gate = (_deq(*t["gate"], GS) @ x).half()
    mask = _select(gate.float().abs()[None], c["k"])[0]
    h = _silu_mul(gate.double(), _deq(*t["up"], GS) @ x) * mask
    return h @ _deq(*t["down"], GS), mask.nonzero().flatten().int()


def _rms(x, w, eps=1e-6):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w.double()


def _exact_generate(c, seed):
    t = _decoder_inputs(c, seed)
    H, I, NQ, NKV, hd = c["H"], c["I"], c["NQ"], c["NKV"], c["hd"]
    inv = 1.0 / 1e6 ** (torch.arange(0, hd, 2, dtype=torch.float64, device=_DEV) / hd)
    cache = [None] * c["layers"]
    head = t["embed"]
    if c["int4_head"]:
        w = t["embed"].float().view(c["vocab"], H // GS, GS)
        s = w.abs().amax(-1) / 7.0
        head = ((w / s[..., None]).round().clamp(-7, 7) * s[..., None]).view(c["vocab"], H)

    def rope(x, pos):
        a = pos[:, None, None] * inv
        x1, x2 = x[..., :hd // 2], x[..., hd // 2:]
        return torch.cat([x1 * a.cos() - x2 * a.sin(), x2 * a.cos() + x1 * a.sin()], -1)

    def layers(tokens, p0):
        x = t["embed"][tokens].double()
        T = x.shape[0]
        pos = torch.arange(p0, p0 + T, device=_DEV, dtype=torch.float64)
        for l, L in enumerate(t["layers"]):
            qkv = _rms(x, L["norms"][0]) @ _deq(*L["qkv"], GS).T
            q, k, v = (z.reshape(T, -1, hd) for z in qkv.split([NQ * hd, NKV * hd, NKV * hd], 1))
            q, k = rope(_rms(q, L["norms"][2]), pos), rope(_rms(k, L["norms"][3]), pos)
            if cache[l] is not None:
                k, v = torch.cat([cache[l][0], k]), torch.cat([cache[l][1], v])
            cache[l] = (k, v)
            live = torch.arange(k.shape[0], device=_DEV)[None] <= pos[:, None]
            a = torch.empty(T, NQ, hd, dtype=torch.float64, device=_DEV)
            for h in range(NQ):
                kv = h // (NQ // NKV)
                sc = (q[:, h] @ k[:, kv].T / math.sqrt(hd)).masked_fill(~live, float("-inf"))
                a[:, h] = torch.softmax(sc, 1) @ v[:, kv]
            x = x + a.reshape(T, -1) @ _deq(*L["o"], GS).T
            h3 = _rms(x, L["norms"][1])
            gu = h3 @ _deq(*L["gu"], GS).T
            x = x + _silu_mul(gu[:, :I], gu[:, I:]) @ _deq(*L["down"], GS).T
        return x[-1]

    tokens = list(t["prompt"])
    x = layers(torch.tensor(tokens, device=_DEV), 0)
    for i in range(c["n"]):
        xn = _rms(x, t["final_norm"])
        logits = torch.cat([h.double() @ xn for h in head.split(16384)])
        tokens.append(int(logits.argmax()))
        if i + 1 < c["n"]:
            x = layers(torch.tensor(tokens[-1:], device=_DEV), len(tokens) - 1)
    return dict(tokens=np.array(tokens), logits=logits)


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "gemv":
        g = _gen(seed)
        q, s = _codes(g, c["N"], c["K"], c["gs"], c["bits"])
        return _deq(q, s, c["gs"]) @ _x(g, c["K"]).double()
    if kind == "group":
        return torch.cat([_deq(q, s, GS) @ x.double() for q, s, x, _ in _group_inputs(c, seed)])
    if kind == "topk":
        return _select(_x(_gen(seed), c["n"]).float().abs()[None], c["k"])[0].nonzero().flatten().int()
    if kind == "dip_mlp":
        y, idx = _exact_mlp(c, seed)
        return dict(y=y, idx=idx)
    if kind == "cached_dip_mlp":
        y, idx = _exact_mlp(c, seed)
        return dict(y=y, idx=idx, misses=None)
    if kind == "attention":
        s = prepare(c, seed)
        q, k, v = (s[n].double() for n in "qkv")
        r = c["NQ"] // c["NKV"]
        k, v = (z[:, :c["L"]].repeat_interleave(r, 0) for z in (k, v))
        p = torch.softmax((k @ q[:, :, None])[..., 0] / math.sqrt(c["hd"]), 1)
        return (p[:, None] @ v)[:, 0]
    if kind == "quantize":
        W = torch.randn(c["N"], c["K"], generator=_gen(seed), device=_DEV) * 0.02
        G = -(-c["K"] // c["gs"])
        w = torch.zeros(c["N"], G * c["gs"], dtype=torch.float64, device=_DEV)
        w[:, :c["K"]] = W
        return dict(packed=None, scale=w.view(c["N"], G, c["gs"]).abs().amax(-1) / 7.0)
    # A DIP decoder has no value in 64 bits that a binary16 one comes near: one |gate| on the other side of the
    # threshold swaps a channel, which moves the next layer's gates (0.26 of the logits after 28 layers, measured).
    return _exact_generate(c, seed) if c["mode"] == "dense" else None
