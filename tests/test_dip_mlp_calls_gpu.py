"""dip_mlp, cached_dip_mlp and their launches against the separate operators (gate GEMV, top-k over fp32 |gate|, indexed
up GEMV, SiLU, indexed accumulate), bit for bit: widths off every vector and tile size (rows of the two matrices in one
8-row tile, K no multiple of 32), fewer rows than the down has counters, more channels than the fused selection takes,
and host rows the kernels can and cannot map."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def make(cuda, I, H, gs, seed):
    from soinfer.quant import formats, pack
    from soinfer.runtime import dip

    g = torch.Generator(device=cuda).manual_seed(seed)

    def m():
        q = formats.quantize(torch.randn(I, H, generator=g, device=cuda) * 0.05, formats.QuantConfig(4, "group", gs))
        return pack.pack_int4(q.qweight[:, :H].contiguous())[0], q.scale

    (gw, s0), (uw, s1), (dw, s2) = m(), m(), m()
    return dip.DipMLPWeights(gw, s0, uw, s1, dw, s2, H, gs), torch.randn(H, generator=g, device=cuda).half()


def by_operators(w, x, k):
    from soinfer import ops
    from soinfer.runtime import dip

    gate = ops.gemv_w4a16_group_lop3(w.gate_Wq, w.gate_scale, x, w.hidden_size, w.group_size)
    idx = ops.topk_threshold_select(gate.float().abs(), k)
    u = ops.gemv_w4a16_indexed(w.up_Wq, w.up_scale, idx, x, w.hidden_size, w.group_size)
    h = dip.silu_gate(gate, idx, u)
    return ops.gemv_w4a16_indexed_accumulate(w.down_T_Wq, w.down_T_scale, idx, h, w.hidden_size, w.group_size), idx


@pytest.mark.parametrize("I,H,gs,k", [(512, 256, 128, 200), (517, 264, 32, 1), (5, 4096, 128, 3), (2051, 1000, 64, 1025),
                                      (4100, 2048, 128, 4100), (8200, 512, 128, 4000)])
def test_dip_mlp_equals_the_operators(cuda, I, H, gs, k):
    from soinfer.offload.hot_cache import HotCache
    from soinfer.runtime import dip

    w, x = make(cuda, I, H, gs, I + k)
    y, idx = by_operators(w, x, k)
    for _ in range(2):  # the counters of the first call are not left behind for the second
        got = dip.dip_mlp(w, x, k)
        assert torch.equal(got[0], y) and torch.equal(got[1], idx)
    hot = list(range(0, I, 3))
    cache = HotCache.build(w.up_Wq, w.up_scale, w.down_T_Wq, w.down_T_scale, hot)
    misses = int((idx % 3 != 0).sum())
    row = w.up_Wq.shape[1]
    pinned = [torch.empty(t.shape, dtype=torch.uint8, pin_memory=True).copy_(t) for t in (w.up_Wq, w.down_T_Wq)]
    staging = torch.empty(k * row, dtype=torch.uint8, pin_memory=True)
    small = torch.empty(max(1, misses) * row, dtype=torch.uint8, pin_memory=True)  # enough for the gathers only
    for host in ((), (*pinned, staging), (*pinned, small)):
        record = []
        got = dip.cached_dip_mlp(w, cache, x, k, *host, miss_bytes=record)
        assert torch.equal(got[0], y) and torch.equal(got[1], idx) and got[2] == misses
        assert record == [2 * misses * row]
    got = dip.cached_dip_mlp_direct(w, cache, x, k, *pinned)
    assert torch.equal(got[0], y) and torch.equal(got[1], idx)


def test_refusals(cuda):
    from soinfer.offload.hot_cache import HotCache
    from soinfer.runtime import dip

    w, x = make(cuda, 64, 128, 64, 1)
    cache = HotCache.build(w.up_Wq, w.up_scale, w.down_T_Wq, w.down_T_scale, [0, 5])
    for k in (0, 65):
        with pytest.raises(RuntimeError):
            dip.dip_mlp(w, x, k)
        with pytest.raises(RuntimeError):
            dip.cached_dip_mlp(w, cache, x, k)
    with pytest.raises(RuntimeError):
        dip.dip_mlp(w, x[:64], 8)
    with pytest.raises(RuntimeError):
        dip.dip_mlp(w, x.float(), 8)
    pinned = [torch.empty(t.shape, dtype=torch.uint8, pin_memory=True).copy_(t) for t in (w.up_Wq, w.down_T_Wq)]
    tiny = torch.empty(16, dtype=torch.uint8, pin_memory=True)
    with pytest.raises(RuntimeError):  # too small for the missing rows
        dip.cached_dip_mlp(w, cache, x, 32, *pinned, tiny)
    with pytest.raises(RuntimeError):  # not pinned
        dip.cached_dip_mlp(w, cache, x, 32, *[p.clone() for p in pinned], tiny)


def test_host_rows_belong_to_the_caller_after_the_call(cuda):
    from soinfer.offload.hot_cache import HotCache
    from soinfer.runtime import dip

    w, x = make(cuda, 4096, 2048, 128, 9)
    y, idx = by_operators(w, x, 4096)
    cache = HotCache.build(w.up_Wq, w.up_scale, w.down_T_Wq, w.down_T_scale, [7])
    pinned = [torch.empty(t.shape, dtype=torch.uint8, pin_memory=True).copy_(t) for t in (w.up_Wq, w.down_T_Wq)]
    staging = torch.empty(pinned[0].numel(), dtype=torch.uint8, pin_memory=True)
    got = dip.cached_dip_mlp(w, cache, x, 4096, *pinned, staging)
    for p in pinned:  # 8 MB of misses take far longer over the link than this
        p.zero_()
    assert torch.equal(got[0], y) and torch.equal(got[1], idx)


@pytest.mark.parametrize("side", ["up", "down"])
def test_a_call_that_fails_leaves_nothing_running(cuda, side):
    """A cache whose rows do not fit fails after the first launches of the call: by the time the error is raised they have
    run, so the miss count's pinned word and the caller's host rows are free."""
    import dataclasses

    from soinfer.offload.hot_cache import HotCache
    from soinfer.runtime import dip

    w, x = make(cuda, 4096, 2048, 128, 9)
    cache = HotCache.build(w.up_Wq, w.up_scale, w.down_T_Wq, w.down_T_scale, [7, 9])
    name = {"up": "up_Wq", "down": "down_Wq"}[side]
    bad = dataclasses.replace(cache, **{name: getattr(cache, name)[:, :-4].contiguous()})
    pinned = [torch.empty(t.shape, dtype=torch.uint8, pin_memory=True).copy_(t) for t in (w.up_Wq, w.down_T_Wq)]
    staging = torch.empty(pinned[0].numel(), dtype=torch.uint8, pin_memory=True)
    for host in ((), (*pinned, staging)):
        torch.cuda.synchronize()
        torch.cuda._sleep(20_000_000)  # the launches of the call wait behind this
        with pytest.raises(RuntimeError):
            dip.cached_dip_mlp(w, bad, x, 4096, *host)
        assert torch.cuda.current_stream().query()
    y, idx = by_operators(w, x, 4096)
    got = dip.cached_dip_mlp(w, cache, x, 4096, *pinned, staging)
    assert torch.equal(got[0], y) and torch.equal(got[1], idx)


@pytest.mark.parametrize("I,k", [(512, 200), (9000, 4000)])
def test_channel_counts_of_gates_that_are_not_numbers(cuda, I, k):
    """Fewer than k gates that are numbers: those channels count once, the rest of the list nothing (the fused selection
    and the separate one above its widths)."""
    from soinfer.runtime import dip

    w, x = make(cuda, I, 256, 128, I)
    counts = torch.zeros(I, dtype=torch.int64, device=cuda)
    _, idx = dip.dip_mlp(w, x, k, counts)
    assert torch.equal(counts.nonzero().flatten(), idx.long()) and int(counts.max()) == 1
    few = torch.arange(3, I, 7, device=cuda)[:k // 3]
    scale = torch.full_like(w.gate_scale, float("nan"))
    scale[few] = w.gate_scale[few]
    w.gate_scale = scale
    counts.zero_()
    _, idx = dip.dip_mlp(w, x, k, counts)
    assert torch.equal(counts.nonzero().flatten(), few) and int(counts.sum()) == few.numel()
    assert torch.equal(idx[:few.numel()].long(), few)
    counts.zero_()
    dip.dip_mlp(w, torch.full_like(x, float("nan")), k, counts)
    assert int(counts.sum()) == 0
