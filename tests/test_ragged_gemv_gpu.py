"""GEMVs over rows of any length and alignment: bit for bit the aligned kernel's result on the same values with the rows
padded by zeros to a multiple of 32 elements (same chunks, same order; zeros add nothing), for row tails of every size,
lengths at and around one and several 64-chunk passes, matrices and vectors off every 16-byte boundary, and the single,
indexed, batched and grouped forms."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops(cuda):
    from soinfer import ops

    return ops


def codes(N, K, gs, bits, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    top = (1 << (bits - 1)) - 1
    q = torch.randint(-top - 1, top + 1, (N, K), generator=g, device="cuda", dtype=torch.int8)
    s = torch.rand(N, -(-K // gs), generator=g, device="cuda") * 0.02 + 1e-3
    return q, s, torch.randn(K, generator=g, device="cuda").half()


def padded(q, x):
    N, K = q.shape
    P = -(-K // 32) * 32
    qp = torch.zeros(N, P, dtype=q.dtype, device="cuda")
    xp = torch.zeros(P, dtype=x.dtype, device="cuda")
    qp[:, :K], xp[:K] = q, x
    return qp, xp


def off(t, nbytes):
    """t's values `nbytes` past an allocation's start."""
    b = torch.empty(t.numel() * t.element_size() + 64, dtype=torch.uint8, device=t.device)
    v = b[nbytes:nbytes + t.numel() * t.element_size()].view(t.dtype).view(t.shape)
    v.copy_(t)
    return v


KS = [32, 33, 39, 40, 47, 48, 56, 57, 63, 100, 300, 1031, 2047, 2049, 2080, 3000, 4100, 6152, 9001]


@pytest.mark.parametrize("K", KS)
@pytest.mark.parametrize("N,gs", [(1, 32), (7, 128), (2050, 8), (4104, 64)])
def test_int4(ops, N, K, gs):
    from soinfer.quant import pack

    q, s, x = codes(N, K, gs, 4, N + K)
    qp, xp = padded(q, x)
    W, Wp = pack.pack_int4(q)[0], pack.pack_int4(qp)[0]
    sp = s if gs >= 32 else torch.cat([s, s.new_zeros(N, Wp.shape[1] * 2 // gs - s.shape[1])], 1).contiguous()
    want = ops.gemv_w4a16_group_lop3(Wp, sp, xp, Wp.shape[1] * 2, gs)
    for fn in (ops.gemv_w4a16_group_lop3, ops.gemv_w4a16_group):
        assert torch.equal(fn(W, s, x, K, gs), want)
    assert torch.equal(ops.gemv_w4a16_group_lop3(off(W, 4), s, off(x, 2), K, gs), want)
    assert torch.equal(ops.gemv_w4a16_group_lop3(off(Wp, 8), sp, xp, Wp.shape[1] * 2, gs), want)
    idx = torch.arange(N - 1, -1, -1, dtype=torch.int32, device="cuda")
    assert torch.equal(ops.gemv_w4a16_indexed(W, s, idx, x, K, gs), want.flip(0))
    assert all(torch.equal(y, want) for y in ops.GemvBatch([W, W.clone()], [s, s], [x, x.clone()], K, gs).run())
    if gs >= 32:
        ys = ops.GemvGroup([(W, s, x, K), (Wp, sp, xp, Wp.shape[1] * 2)], gs).run()
        assert torch.equal(ys[0], want) and torch.equal(ys[1], want)


@pytest.mark.parametrize("K", [16, 17, 31] + KS)
@pytest.mark.parametrize("N,gs", [(1, 32), (9, 128), (4100, 16), (17000, 4)])
def test_int8(ops, N, K, gs):
    q, s, x = codes(N, K, gs, 8, N + K)
    qp, xp = padded(q, x)
    P = qp.shape[1]
    sp = torch.cat([s, s.new_zeros(N, -(-P // gs) - s.shape[1])], 1).contiguous()
    want = ops.gemv_w8a16(qp, sp, xp, gs)
    assert torch.equal(ops.gemv_w8a16(q, s, x, gs), want)
    assert torch.equal(ops.gemv_w8a16(off(q, 3), s, off(x, 2), gs), want)
    assert torch.equal(ops.gemv_w8a16(off(qp, 5), sp, xp, gs), want)
    assert all(torch.equal(y, want) for y in ops.Int8Batch([q, q.clone()], [s, s], [x, x.clone()], gs).run())
    one = s[:, :1].contiguous()  # one scale per row
    assert torch.equal(ops.gemv_w8a16(q, one, x, K), ops.gemv_w8a16(qp, one, xp, P))


@pytest.mark.parametrize("K", [2560, 4096, 5120, 6144, 8192])
@pytest.mark.parametrize("N", [2049, 4096, 4100, 6145, 8191, 8192, 8198, 12287, 24577])
def test_int4_rows_per_wave(ops, N, K):
    """Every line of the rows-per-wave rule (2 and 4 rows, their remainders): a row's result does not depend on its tile,
    so it is the one-row tile's of the same rows in matrices of under 2048."""
    from soinfer.quant import pack

    q, s, x = codes(N, K, 128, 4, N + K)
    W = pack.pack_int4(q)[0]
    got = ops.gemv_w4a16_group_lop3(W, s, x, K, 128)
    for r in range(0, N, 1024):
        part = slice(r, min(N, r + 1024))
        assert torch.equal(got[part], ops.gemv_w4a16_group_lop3(W[part], s[part], x, K, 128))
