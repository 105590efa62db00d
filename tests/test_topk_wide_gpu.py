"""top-k at the edges of its kernels' ranges (8 and 16 waves, 24 and 32 values a lane, the streamed form), with ties, zeros
and a huge value, against the reference rule."""
import numpy as np
import pytest
import torch

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [16383, 16384, 16385, 17408, 24575, 24576, 24577, 27648, 32767, 32768, 32769])
@pytest.mark.parametrize("frac", [0.0, 0.3, 1.0])
def test_wide_selection(cuda, n, frac):
    from soinfer import ops

    k = max(1, int(n * frac))
    g = np.abs(np.random.default_rng(n + k).standard_normal(n)).astype(np.float32)
    g[::7] = g[3]  # a seventh of the values tie
    g[1::11] = 0.0
    g[5] = np.float32(1e30)
    got = ops.topk_threshold_select(torch.from_numpy(g).to(cuda), k)
    assert np.array_equal(got.cpu().numpy(), O.topk_rule_a(g, k))


@pytest.mark.parametrize("n", [16384, 16385, 17408, 24576, 24577, 32768, 32769])
@pytest.mark.parametrize("frac", [0.0, 0.3, 1.0])
def test_wide_selection_of_binary16_gates(cuda, n, frac):
    """The |gate| form of the same kernels (what a 17408-wide engine selects with): signs, ties, infinities, and NaN (never
    selected: with every channel asked for, fewer than k are)."""
    from soinfer import _C

    k = max(1, int(n * frac))
    gate = torch.randn(n, generator=torch.Generator().manual_seed(n + k)).half()
    gate[::7], gate[1::11], gate[5], gate[9] = gate[3].clone(), 0.0, float("inf"), float("-inf")
    gate[13::101] = float("nan")
    want = O.topk_rule_a(gate.float().abs().numpy(), k)
    idx = torch.full((k,), -7, dtype=torch.int32, device=cuda)
    cnt = torch.zeros(1, dtype=torch.int32, device=cuda)
    _C.topk_threshold_select_f16abs_into(gate.to(cuda), k, idx, cnt)
    assert int(cnt) == want.size
    assert np.array_equal(idx.cpu().numpy()[:want.size], want) and bool((idx[want.size:] == -7).all())
