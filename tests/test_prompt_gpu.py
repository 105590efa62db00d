"""A whole prompt through the layers together against the same tokens one at a time: every token's K and V, the final
hidden state, its norm and the first generated token bit for bit, at the edges of the token tiles (4 and 8 tokens),
contexts past one attention workgroup's rows (split plan), ragged widths (hidden and attention widths that are no
multiple of 2048 elements; the one-pass norm at hidden 2048), group sizes 32 to 128, a second prompt appended to the
first, and streamed weights. The matrix-core products (dense prompts of PROMPT_MFMA tokens up) sum in another order:
each is held to the binary64 product of the same operands, and the engine's state to the one-at-a-time state."""
import ctypes
from pathlib import Path

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dec(cuda):
    from soinfer.runtime import decoder

    return decoder


CONFIGS = {
    "h256": dict(hidden=256, q_heads=4, kv_heads=2, head_dim=64, intermediate=512, group_size=128),
    "h2048": dict(hidden=2048, q_heads=16, kv_heads=8, head_dim=128, intermediate=1024, group_size=128),
    "h416_gs32": dict(hidden=416, q_heads=3, kv_heads=1, head_dim=32, intermediate=352, group_size=32),
    "h2176_gs64": dict(hidden=2176, q_heads=8, kv_heads=1, head_dim=64, intermediate=2240, group_size=64),
}


@pytest.fixture(scope="module", params=list(CONFIGS))
def weights(request, dec):
    cfg = dec.DecoderConfig(layers=2, vocab=1000, max_seq=640, **CONFIGS[request.param])
    return dec.random_decoder(cfg, seed=7, linear_std=0.05, norm_jitter=0.1)


@pytest.fixture
def in_order(dec, monkeypatch):
    """Prompts of every length in the decode step's order of operations."""
    monkeypatch.setattr(dec, "PROMPT_MFMA", 1 << 30)


def tokens(n, vocab, seed):
    return torch.randint(0, vocab, (n,), generator=torch.Generator().manual_seed(seed)).tolist()


def one_at_a_time(eng, prompt):
    for t in prompt:
        eng.token.fill_(t)
        eng._layers()


def same_state(a, b, n, what):
    for l in range(a.c.layers):
        assert torch.equal(a.k_cache[l][:, :n], b.k_cache[l][:, :n]), f"{what}: layer {l} K"
        assert torch.equal(a.v_cache[l][:, :n], b.v_cache[l][:, :n]), f"{what}: layer {l} V"
    assert torch.equal(a.x_final, b.x_final), f"{what}: hidden state"
    assert torch.equal(a.hn, b.hn), f"{what}: final norm"
    assert torch.equal(a.pos, b.pos) and torch.equal(a.token, b.token), f"{what}: position or token"


@pytest.mark.parametrize("n", [3, 4, 5, 8, 9, 33, 301])
def test_prompt_equals_single_steps(dec, weights, in_order, n):
    a = dec.DecodeEngine(weights, "dense", max_new_tokens=2)
    b = dec.DecodeEngine(weights, "dense", max_new_tokens=2)
    prompt = tokens(n, weights.config.vocab, n)
    for e in (a, b):
        e.reset()
    assert a._prompt_together(n)
    a.prefill(prompt, use_graph=False)
    one_at_a_time(b, prompt)
    same_state(a, b, n, f"{n} tokens")
    more = tokens(6, weights.config.vocab, n + 1)  # a second prompt behind the first
    a.prefill(more, use_graph=False)
    one_at_a_time(b, more)
    same_state(a, b, n + 6, f"{n} + 6 tokens")
    for e in (a, b):
        e.decode(2, use_graph=False)
    assert torch.equal(a.log, b.log) and torch.equal(a.logits, b.logits)


def test_streamed_prompt_equals_resident(dec, weights):
    prompt = tokens(20, weights.config.vocab, 3)
    a = dec.DecodeEngine(weights, "dense", max_new_tokens=4)
    want = a.generate(prompt, 4)
    for overlap in (True, False):
        e = dec.DecodeEngine(weights, "dense", max_new_tokens=4, offload=True, overlap_copy=overlap)
        for _ in range(2):
            assert e.generate(prompt, 4) == want
            same_state(a, e, 24, f"overlap {overlap}")


def dip_engines(dec, w, k):
    hot = [list(range(0, w.config.intermediate, 3)) for _ in range(w.config.layers)]
    none = [[] for _ in range(w.config.layers)]
    return {"indexed": dict(mode="dip", dip_schedule="indexed"), "default": dict(mode="dip"),
            "gated": dict(mode="dip", dip_schedule="gated"),
            "cached": dict(mode="cached_dip", hot_channels=hot),
            "all missing": dict(mode="cached_dip", hot_channels=none, miss_path="staged"),
            "streamed": dict(mode="cached_dip", hot_channels=hot, offload=True)}


@pytest.mark.parametrize("n,frac", [(3, 0.5), (9, 0.02), (33, 0.9), (301, 0.5), (4, 1.0)])
def test_dip_prompt_equals_single_steps(dec, weights, n, frac):
    """DIP: one selected channel per 50 (a row chunk of a few rows) up to all of them (several row chunks and their
    remainder), resident and cache-aware. The selections agree where the hidden states do."""
    c = weights.config
    k = max(1, int(c.intermediate * frac))
    prompt, more = tokens(n, c.vocab, n), tokens(5, c.vocab, n + 1)
    for what, kw in dip_engines(dec, weights, k).items():
        a, b = (dec.DecodeEngine(weights, dip_k=k, max_new_tokens=2, **kw) for _ in range(2))
        for e in (a, b):
            e.reset()
        assert a._prompt_together(n)
        for part, total in ((prompt, n), (more, n + 5)):
            a.prefill(part, use_graph=False)
            one_at_a_time(b, part)
            same_state(a, b, total, f"{what}, {total} tokens")


def test_calibration_counts_of_a_prompt(dec, weights):
    c = weights.config
    prompt, k = tokens(21, c.vocab, 5), c.intermediate // 3
    a, b = (dec.DecodeEngine(weights, "dip", dip_k=k, max_new_tokens=1) for _ in range(2))
    for e in (a, b):
        e.counts = [torch.zeros(c.intermediate, dtype=torch.int64, device="cuda") for _ in range(c.layers)]
        e.reset()
    a.prefill(prompt, use_graph=False)
    one_at_a_time(b, prompt)
    for l in range(c.layers):
        assert torch.equal(a.counts[l], b.counts[l]) and int(a.counts[l].sum()) == 21 * k


@pytest.mark.parametrize("n", [9, 16, 17, 65, 301])
def test_matrix_core_prompt_near_single_steps(dec, weights, n):
    """Each linear's binary16 result can move to a neighbour (2^-11), which the following layers carry: after two
    layers the states stay within 1% of their largest element (the decode engine's own bound against the oracle on
    such models is half of that on logits, which average the state)."""
    a = dec.DecodeEngine(weights, "dense", max_new_tokens=2)
    b = dec.DecodeEngine(weights, "dense", max_new_tokens=2)
    prompt = tokens(n, weights.config.vocab, n)
    for e in (a, b):
        e.reset()
    a.prefill(prompt)
    one_at_a_time(b, prompt)
    near_state(a, b, n)


@pytest.mark.parametrize("what", ["dense", "default", "indexed", "cached", "streamed"])
def test_prompt_in_parts(dec, weights, monkeypatch, what):
    """A prompt longer than one part: parts of 16, 16 and 1 tokens, the later ones behind a context (dense: the first two
    on the matrix cores, the last in the step's order)."""
    monkeypatch.setattr(dec, "PROMPT_CHUNK", 16)
    c = weights.config
    kw = dict(mode="dense") if what == "dense" else dict(dip_k=c.intermediate // 2,
                                                         **dip_engines(dec, weights, 1)[what])
    a, b = (dec.DecodeEngine(weights, max_new_tokens=2, **kw) for _ in range(2))
    prompt = tokens(33, c.vocab, 11)
    for e in (a, b):
        e.reset()
    a.prefill(prompt)
    one_at_a_time(b, prompt)
    b.token.fill_(prompt[-1])
    if what != "dense":
        same_state(a, b, 33, what)
        return
    near_state(a, b, 33)


def near_state(a, b, n):
    pairs = [(a.x_final, b.x_final), (a.hn, b.hn)]
    for l in range(2):
        pairs += [(a.k_cache[l][:, :n], b.k_cache[l][:, :n]), (a.v_cache[l][:, :n], b.v_cache[l][:, :n])]
    for x, y in pairs:
        x, y = x.float(), y.float()
        assert (x - y).abs().max() <= 1e-2 * y.abs().max()
    assert torch.equal(a.pos, b.pos)


def fragments(x):
    """x [T, K] in the layout soi_gemm_w4a16_mfma reads (tokens rounded up to 16; the rest NaN: never read into a
    result)."""
    T, K = x.shape
    z = torch.full((-(-T // 16) * 16, K), float("nan"), dtype=x.dtype, device=x.device)
    z[:T] = x
    return z.view(-1, 16, K // 128, 4, 4, 8).permute(0, 2, 4, 3, 1, 5).contiguous()


@pytest.mark.parametrize("N,K,gs", [(4, 128, 128), (20, 256, 256), (136, 1152, 128), (256, 1024, 128), (4096, 384, 384),
                                    (2048, 6144, 128)])
@pytest.mark.parametrize("T", [1, 16, 17, 33, 64, 65, 200])
def test_matrix_core_linear(cuda, N, K, gs, T):
    """Tiles of 16 and 32 rows (N below, at and past each), one to four token tiles and their remainders, 4 and 8 waves
    over 1 to 48 steps, scale groups of 1 to 3 steps."""
    check_matrix_core_linear(cuda, N, K, gs, T)


@pytest.mark.parametrize("N,K,T", [(12288, 256, 200), (12308, 384, 193), (33024, 256, 16), (33024, 128, 32)])
def test_matrix_core_linear_of_64_row_tiles(cuda, N, K, T):
    """The tiles of launches of 2048 16-row x token tiles up, over one, two and four token tiles, N with and without a
    remainder."""
    check_matrix_core_linear(cuda, N, K, 128, T)


@pytest.mark.parametrize("scale", [1e-5, 3e-7])
def test_matrix_core_linear_of_subnormal_activations(cuda, scale):
    check_matrix_core_linear(cuda, 256, 1024, 128, 33, scale)


def check_matrix_core_linear(cuda, N, K, gs, T, x_scale=1.0):
    """Every epilogue against binary64. The sum of K products in binary32 is within K 2^-24 of the sum of their absolute
    values; the result is then rounded to binary16."""
    from soinfer.quant import formats, pack

    lib = ctypes.CDLL(str(Path(pack.__file__).resolve().parent.parent / "libsoinfer_hip.so"))
    g = torch.Generator(device=cuda).manual_seed(N + K + T)
    qt = formats.quantize(torch.randn(N, K, generator=g, device=cuda) * 0.02, formats.QuantConfig(4, "group", gs))
    W = pack.pack_int4(qt.qweight)[0].contiguous()
    x = (torch.randn(T, K, generator=g, device=cuda) * x_scale).half()
    w64 = (qt.qweight.double().view(N, K // gs, gs) * qt.scale.double()[..., None]).view(N, K)
    ref, mag = x.double() @ w64.T, x.double().abs() @ w64.abs().T
    bound = K * 2.0 ** -24 * mag + 2.0 ** -11 * ref.abs() + 2.0 ** -24

    def run(y, epilogue):
        st = lib.soi_gemm_w4a16_mfma(*(ctypes.c_void_p(t.data_ptr()) for t in (W, qt.scale, fragments(x), y)),
                                     *(ctypes.c_int64(v) for v in (N, K, gs, T)), ctypes.c_int(epilogue),
                                     ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
        torch.cuda.synchronize()
        return st

    y = torch.full((T + 1, N), 7.0, dtype=torch.float16, device=cuda)
    assert run(y, 0) == 0
    assert bool(((y[:T].double() - ref).abs() <= bound).all())
    assert bool((y[T] == 7.0).all()), "rows past the last token are untouched"
    r = torch.randn(T, N, generator=g, device=cuda).half()
    added = r.clone()
    assert run(added, 1) == 0
    assert torch.equal(added, r + y[:T]), "the residual form adds the same product once, in binary16"
    h = torch.full((-(-T // 16) * 16 * (N // 2),), 7.0, dtype=torch.float16, device=cuda)
    if N % 256:
        assert run(h, 2) != 0, "the fragment layout of the gated output needs N / 2 a multiple of 128"
        return
    assert run(h, 2) == 0
    t = y[:T].view(T, N // 8, 2, 4).float()
    gate, up = t[:, :, 0], t[:, :, 1]
    want = (gate / (1 + torch.exp(-gate)) * up).view(T, N // 2)
    got = h.view(-1, N // 256, 4, 4, 16, 8).permute(0, 4, 1, 3, 2, 5).reshape(-1, N // 2)[:T].float()
    assert bool(((got - want).abs() <= 2.0 ** -10 * want.abs() + 2.0 ** -24).all())


def hip_lib():
    from soinfer.quant import pack

    return ctypes.CDLL(str(Path(pack.__file__).resolve().parent.parent / "libsoinfer_hip.so"))


@pytest.mark.parametrize("n,k", [(512, 200), (6144, 3072), (16384, 16384)])
def test_selection_of_gates_that_are_not_numbers(cuda, n, k):
    """A token with m < k gates that are numbers selects those and leaves -1 in the rest of its list and no mark; the
    other tokens' lists are those of the same gates without it."""
    g = torch.Generator(device=cuda).manual_seed(n)
    gate = torch.randn(4, n, generator=g, device=cuda).half()
    gate[1] = float("nan")
    m = max(1, k // 3)
    numbers = torch.randperm(n, generator=g, device=cuda)[:m].sort().values
    kept = gate[2, numbers].clone()
    gate[2] = float("nan")
    gate[2, numbers] = kept
    idx = torch.full((4, k), 12345678, dtype=torch.int32, device=cuda)
    mark = torch.zeros(n, dtype=torch.int32, device=cuda)
    last = [torch.full((s,), 77, dtype=torch.int32, device=cuda) for s in (k, 1)]
    ptr = [ctypes.c_void_p(t.data_ptr()) for t in (gate, idx, mark, *last)]
    st = hip_lib().soi_dip_select_tokens(ptr[0], *(ctypes.c_int64(v) for v in (n, n, k, 4)), ptr[1], ptr[2],
                                         ctypes.c_int32(9), *ptr[3:], ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert st == 0
    from soinfer import ops

    for t in (0, 3):
        assert torch.equal(idx[t], ops.topk_threshold_select(gate[t].float().abs(), k))
    assert bool((idx[1] == -1).all())
    assert torch.equal(idx[2, :m].long(), numbers) and bool((idx[2, m:] == -1).all())
    named = torch.zeros(n, dtype=torch.bool, device=cuda)
    for t in (0, 2, 3):
        named[idx[t][idx[t] >= 0].long()] = True
    assert torch.equal(mark == 9, named)
    assert torch.equal(last[0], idx[3]) and int(last[1]) == k
    st = hip_lib().soi_dip_select_tokens(ptr[0], *(ctypes.c_int64(v) for v in (n, n, k, 3)), ptr[1], None,
                                         ctypes.c_int32(0), *ptr[3:], ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert st == 0 and int(last[1]) == m
    assert torch.equal(last[0][:m].long(), numbers) and torch.equal(last[0][m:], idx[3, m:]), "nothing past the count"


def test_calibration_counts_of_a_token_without_numbers(dec, weights):
    """A token whose hidden state is not a number selects nothing: the counts are the other tokens'. (Last in the prompt:
    tokens after it attend to its K and V.)"""
    import dataclasses

    c = weights.config
    embed = weights.embed.clone()
    embed[5] = float("nan")
    w = dataclasses.replace(weights, embed=embed)
    k = c.intermediate // 3
    prompt = [t if t != 5 else 6 for t in tokens(21, c.vocab, 5)]
    want = dec.calibrate_channel_counts(w, k, prompt)
    got = dec.calibrate_channel_counts(w, k, prompt + [5])
    for a, b in zip(got, want):
        assert torch.equal(a, b) and int(b.sum()) == 21 * k


@pytest.mark.parametrize("mode", ["dense", "dip", "cached_dip"])
def test_scratch_given_back_while_another_stream_uses_it(cuda, dec, weights, mode):
    """A prompt waits on a side stream while the scratch, which belongs to the default stream, is grown there and its old
    memory is handed out again and overwritten: the prompt's state is that of an undisturbed one."""
    c = weights.config
    kw = {} if mode == "dense" else dict(dip_k=c.intermediate // 2)
    if mode == "cached_dip":
        kw["hot_channels"] = [list(range(0, c.intermediate, 3))] * c.layers
    e = dec.DecodeEngine(weights, mode, max_new_tokens=1, **kw)
    prompt = torch.tensor(tokens(16, c.vocab, 8), dtype=torch.int32, device=cuda)
    e.reset()
    e._prompt_layers(prompt)
    want = e.x_final.clone()
    sizes = [t.numel() * t.element_size() for v in e._prompt_buf.values() for t in (v if isinstance(v, list) else [v])
             if isinstance(t, torch.Tensor)]
    e.reset()
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        torch.cuda._sleep(100_000_000)
        e._prompt_layers(prompt)
    e._prompt_scratch(200)
    taken = [torch.full((n,), 255, dtype=torch.uint8, device=cuda) for n in sizes]
    assert not side.query(), "the prompt is still waiting"
    side.synchronize()
    assert torch.equal(e.x_final, want)
    del taken


@pytest.mark.parametrize("mode,name", [("dense", "o_Wq"), ("dense", "down_Wq"), ("dip", "o_Wq"), ("dip", "down_T_Wq")])
def test_prompt_over_rows_off_16_bytes(cuda, dec, weights, mode, name):
    """The decode step takes the down and down^T rows, and without the deferred attention combine the o rows, from any
    address, so a prompt does too."""
    import dataclasses

    def off(t):
        b = torch.empty(t.numel() + 16, dtype=t.dtype, device=t.device)
        return b[4:4 + t.numel()].view(t.shape).copy_(t)

    c = weights.config
    kw = dict(dip_k=None if mode == "dense" else c.intermediate // 2, defer_attention_combine=name != "o_Wq")
    moved = dataclasses.replace(weights, layers=[dataclasses.replace(L, **{name: off(getattr(L, name))})
                                                 for L in weights.layers])
    prompt = tokens(7, c.vocab, 4)
    a = dec.DecodeEngine(moved, mode, max_new_tokens=3, **kw)
    b = dec.DecodeEngine(weights, mode, max_new_tokens=3, **kw)
    for use_graph in (False, True):
        assert a.generate(prompt, 3, use_graph=use_graph) == b.generate(prompt, 3, use_graph=use_graph)
        same_state(a, b, 10, f"{mode} {name}")


def test_short_prompts_behind_a_context(cuda, dec, weights):
    """The engine counts the tokens behind it, and a short prompt's state is the single steps' on either route."""
    c = weights.config
    for mode, kw in (("dense", {}), ("dip", dict(dip_k=c.intermediate // 2))):
        a = dec.DecodeEngine(weights, mode, max_new_tokens=4, **kw)
        b = dec.DecodeEngine(weights, mode, max_new_tokens=4, **kw)
        a.generate(tokens(5, c.vocab, 1), 3)
        assert a._context == int(a.pos) == 8
        for e in (a, b):
            e.reset()
        total = 0
        for n, apart in ((3, False), (4, True), (2, False), (5, False), (3, True)):
            part = tokens(n, c.vocab, total)
            assert a._prompt_together(n, a._graph_layers is not None) == (n > 2)
            if apart:
                a._prompt_together = lambda *_: False
            a.prefill(part, use_graph=a._graph_layers is not None)
            a.__dict__.pop("_prompt_together", None)
            one_at_a_time(b, part)
            total += n
            same_state(a, b, total, f"{mode}, {total} tokens")
            assert a._context == int(a.pos) == total
        a.decode(2)
        assert a._context == int(a.pos) == total + 2
        a._context = 1 << 30
        assert mode == "dip" or a._prompt_together(9)
        assert a._prompt_together(3, use_graph=False), "eager steps are slower"
    b.reset()
    b.prefill(tokens(3, c.vocab, 7))  # no graph captured
    assert int(b.pos) == 3


@pytest.mark.parametrize("mode", ["dense", "dip", "cached_dip"])
@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
def test_a_token_that_is_not_a_number_leaves_the_others_alone(cuda, dec, weights, mode, bad):
    """Its hidden state is not a number; the K and V of the tokens before it are those of the prompt without it."""
    import dataclasses

    c = weights.config
    embed = weights.embed.clone()
    embed[5, ::3] = bad
    w = dataclasses.replace(weights, embed=embed)
    kw = {} if mode == "dense" else dict(dip_k=c.intermediate // 2)
    if mode == "cached_dip":
        kw["hot_channels"] = [list(range(0, c.intermediate, 3))] * c.layers
    a, b = (dec.DecodeEngine(w, mode, max_new_tokens=1, **kw) for _ in range(2))
    prompt = [t if t != 5 else 6 for t in tokens(20, c.vocab, 5)]
    for e, p in ((a, prompt + [5]), (b, prompt)):
        e.reset()
        e.prefill(p, use_graph=False)
    assert not bool(torch.isfinite(a.x_final).any())
    for l in range(c.layers):
        assert torch.equal(a.k_cache[l][:, :20], b.k_cache[l][:, :20])
        assert torch.equal(a.v_cache[l][:, :20], b.v_cache[l][:, :20])
        assert bool(torch.isfinite(b.k_cache[l][:, :20]).all())
