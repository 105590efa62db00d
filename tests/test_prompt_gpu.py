"""A whole prompt through the layers together against the same tokens one at a time: every token's K and V, the final
hidden state, its norm and the first generated token bit for bit, at the edges of the token tiles (4 and 8 tokens),
contexts past one attention workgroup's rows (split plan), ragged widths (hidden and attention widths that are no
multiple of 2048 elements; the one-pass norm at hidden 2048), group sizes 32 to 128, a second prompt appended to the
first, and streamed weights."""
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


@pytest.mark.parametrize("n", [2, 4, 5, 8, 9, 33, 301])
def test_prompt_equals_single_steps(dec, weights, n):
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
