"""The default DIP engine (no schedule named) against the named indexed schedule: tokens, hidden states, logits and caches
bit for bit, eager and graph replays, where the gated launches run (one- and many-pass norms, the ordered and the row form
of the down) and where they do not fit; and a layer hook sees the indexed schedule's buffers."""
import pytest
import torch

pytestmark = pytest.mark.gpu

CONFIGS = {
    "ordered": (dict(hidden=256, q_heads=4, kv_heads=2, head_dim=64, intermediate=512), 200, True),
    "one_pass": (dict(hidden=2048, q_heads=4, kv_heads=2, head_dim=128, intermediate=1536), 700, True),
    "row_form": (dict(hidden=512, q_heads=4, kv_heads=2, head_dim=64, intermediate=9216), 6000, True),
    "row_form_only": (dict(hidden=512, q_heads=4, kv_heads=2, head_dim=64, intermediate=9216), 8800, True),
    "too_wide": (dict(hidden=1024, q_heads=4, kv_heads=2, head_dim=64, intermediate=20480), 2000, False),
    "other_norm": (dict(hidden=2048, q_heads=4, kv_heads=2, head_dim=128, intermediate=4100), 900, False),
    "odd_width": (dict(hidden=256, q_heads=4, kv_heads=2, head_dim=64, intermediate=518), 100, False),
}


@pytest.mark.parametrize("name", list(CONFIGS))
def test_default_equals_indexed(cuda, name):
    from soinfer.runtime import decoder as D

    kw, k, fits = CONFIGS[name]
    w = D.random_decoder(D.DecoderConfig(layers=2, vocab=700, max_seq=400, **kw), seed=5, linear_std=0.05,
                         norm_jitter=0.1)
    a = D.DecodeEngine(w, "dip", dip_k=k, max_new_tokens=6)
    b = D.DecodeEngine(w, "dip", dip_k=k, max_new_tokens=6, dip_schedule="indexed")
    assert a._gated_now == fits and not b._gated_now
    prompt = torch.randint(0, 700, (290,), generator=torch.Generator().manual_seed(3)).tolist()
    for n in (1, 2, 290):
        want = b.generate(prompt[:n], 6)
        for use_graph in (False, True):
            assert a.generate(prompt[:n], 6, use_graph=use_graph) == want
            assert torch.equal(a.x_final, b.x_final) and torch.equal(a.logits, b.logits)
            for l in range(2):
                assert torch.equal(a.k_cache[l][:, :n + 6], b.k_cache[l][:, :n + 6])
    seen = {}
    for e in (a, b):
        e.layer_hook = lambda l, e=e: seen.setdefault(id(e), []).append(
            [t.clone() for t in (e.h, e.gu[:kw["intermediate"]], e.idx, e.h_sel, e.down)])
        e._layers()
        e.layer_hook = None
    for x, y in zip(seen[id(a)], seen[id(b)]):
        assert all(torch.equal(p, q) for p, q in zip(x, y))


@pytest.mark.parametrize("name", ["ordered", "one_pass", "row_form_only"])
def test_selection_of_the_latest_step_is_readable(cuda, name):
    """idx and cnt after prompts, single steps and graph replays are the indexed schedule's."""
    from soinfer.runtime import decoder as D

    kw, k, _ = CONFIGS[name]
    w = D.random_decoder(D.DecoderConfig(layers=2, vocab=700, max_seq=400, **kw), seed=5, linear_std=0.05,
                         norm_jitter=0.1)
    a = D.DecodeEngine(w, "dip", dip_k=k, max_new_tokens=6)
    b = D.DecodeEngine(w, "dip", dip_k=k, max_new_tokens=6, dip_schedule="indexed")
    cached = D.DecodeEngine(w, "cached_dip", dip_k=k, max_new_tokens=6,
                            hot_channels=[list(range(0, kw["intermediate"], 3))] * 2)
    prompt = torch.randint(0, 700, (9,), generator=torch.Generator().manual_seed(3)).tolist()

    def same(what):
        assert torch.equal(a.idx, b.idx) and torch.equal(a.cnt, b.cnt), what
        assert torch.equal(cached.idx, b.idx) and torch.equal(cached.cnt, b.cnt), what

    for e in (a, b, cached):
        e.reset()
    b._prompt_together = lambda *_: False
    for e in (a, b, cached):
        e.prefill(prompt, use_graph=False)
    same("prompt")
    for e in (a, b, cached):
        e.decode(1, use_graph=False)
    same("one step")
    for e in (a, b, cached):
        e.generate(prompt, 6)
    same("generate")
