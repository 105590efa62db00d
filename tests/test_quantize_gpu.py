"""The device quantizer and packer against the tensor expressions on the CPU (which the oracle pins): codes, scales and
bytes exactly, over group sizes, bit widths, ragged K, offset views, groups of zeros, denormals, infinities and NaN; and
the calls that have to see the tensor operations still do."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def same(a, b):
    assert a.shape == b.shape and a.dtype == b.dtype
    if a.dtype.is_floating_point:
        a, b = a.view(torch.int32), b.view(torch.int32)
    assert torch.equal(a.cpu(), b.cpu())


@pytest.mark.parametrize("gs", [32, 64, 128, 256])
@pytest.mark.parametrize("N,K", [(1, 1), (3, 31), (5, 128), (7, 257), (64, 2048), (2, 4100), (33, 1000)])
def test_group_quantize_and_pack(cuda, gs, N, K):
    from soinfer.quant import formats, pack

    g = torch.Generator().manual_seed(N * K + gs)
    w = torch.randn(N, K, generator=g) * 0.02
    w[0, : K // 2] = 0.0
    if K > 257:
        w[-1, 0], w[-1, 3], w[-1, gs], w[-1, gs + 1] = 1e-41, -3e-42, 1e38, -3.4e38  # denormal and huge groups
    for bits in (2, 4, 8):
        cfg = formats.QuantConfig(bits, "group", gs)
        want, got = formats.quantize(w, cfg), formats.quantize(w.to(cuda), cfg)
        same(got.qweight, want.qweight)
        same(got.scale, want.scale)
        if bits == 4:
            same(pack.pack_int4(got.qweight)[0], pack.pack_int4(want.qweight)[0])
            same(pack.pack_int4(got.qweight[:, :K])[0], pack.pack_int4(want.qweight[:, :K])[0])  # ragged rows


def test_shapes_and_views(cuda):
    from soinfer.quant import formats, pack

    cfg = formats.QuantConfig(4, "block32")
    base = torch.randn(1 + 2 * 3 * 96, generator=torch.Generator().manual_seed(1))
    for w in (base[1:].view(2, 3, 96), base[1:97], base[1:].view(6, 96).t(), base[:96].half()):
        d = w.to(cuda) if w.is_contiguous() else base.to(cuda)[1:].view(6, 96).t()
        want, got = formats.quantize(w, cfg), formats.quantize(d, cfg)
        same(got.qweight, want.qweight)
        same(got.scale, want.scale)
    d = base.to(cuda)[1:577].view(6, 96)  # 4 bytes past a 16-byte boundary
    same(formats.quantize(d, cfg).qweight, formats.quantize(base[1:577].view(6, 96), cfg).qweight)
    q = torch.randint(-128, 128, (1 + 4 * 64,), generator=torch.Generator().manual_seed(2), dtype=torch.int8)
    same(pack.pack_int4(q.to(cuda)[1:].view(4, 64))[0], pack.pack_int4(q[1:].view(4, 64))[0])  # only low nibbles count
    same(pack.pack_int4(q.to(cuda)[1:])[0], pack.pack_int4(q[1:])[0])


def test_not_finite(cuda):
    """A group with a NaN or an infinity: the expressions' scale and codes on the device."""
    from soinfer.quant import calibrate, formats

    w = torch.randn(4, 256, device=cuda, generator=torch.Generator(device=cuda).manual_seed(3))
    w[0, 5], w[1, 130], w[2, 7] = float("nan"), float("inf"), float("-inf")
    cfg = formats.QuantConfig(4, "group", 128)
    got = formats.quantize(w, cfg)
    want = formats.quantize(w, cfg, lambda *a: calibrate.min_max(*a))  # another function: the tensor expressions
    same(got.scale.nan_to_num(7.0), want.scale.nan_to_num(7.0))
    same(got.qweight, want.qweight)


def test_observed_calls_take_the_expressions(cuda):
    from soinfer.quant import formats

    cfg = formats.QuantConfig(4, "group", 64)
    w = torch.randn(4, 128, device=cuda, requires_grad=True)
    assert formats.quantize(w, cfg).scale.requires_grad
    with torch.no_grad():
        assert not formats.quantize(w, cfg).scale.requires_grad
    plain = w.detach()
    rows = torch.vmap(lambda r: formats.quantize(r, cfg).scale)(plain)
    same(rows, formats.quantize(plain, cfg).scale)


@pytest.mark.parametrize("n,H", [(8, 1), (8, 8), (64, 64), (72, 65), (136, 1000), (6144, 2048)])
def test_transposed_rows(cuda, n, H):
    from soinfer import ops
    from soinfer.quant import pack

    q = torch.randint(-8, 8, (n, H), generator=torch.Generator().manual_seed(n + H), dtype=torch.int8)
    s = torch.rand(n, 3)
    W = pack.pack_int4(q)[0]
    got, gs = ops.transposed_down_T(W.to(cuda), s.to(cuda), H)
    same(got, pack.pack_int4(q.t().contiguous())[0])
    same(gs, s.t().contiguous())


def test_negative_views_and_modes(cuda):
    """A negative view (its negation still to be done) and calls under a dispatch mode take the expressions."""
    from torch.utils._python_dispatch import TorchDispatchMode

    from soinfer import ops
    from soinfer.quant import formats, pack

    cfg = formats.QuantConfig(4, "group", 64)
    w = torch.randn(4, 128, device=cuda, generator=torch.Generator(device=cuda).manual_seed(5))
    want, got = formats.quantize(-w, cfg), formats.quantize(torch._neg_view(w), cfg)
    same(got.qweight, want.qweight)
    same(got.scale, want.scale)
    q = torch.randint(-8, 8, (64, 128), generator=torch.Generator().manual_seed(6), dtype=torch.int8).to(cuda)
    same(pack.pack_int4(torch._neg_view(q))[0], pack.pack_int4(-q)[0])

    class Seen(TorchDispatchMode):
        ops = 0

        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            Seen.ops += 1
            return func(*args, **(kwargs or {}))

    W, s = pack.pack_int4(q)[0], torch.rand(64, 1, device=cuda)
    want = ops.transposed_down_T(W, s, 128)
    with Seen():
        got = ops.transposed_down_T(W, s, 128)
    assert Seen.ops > 5 and all(torch.equal(a, b) for a, b in zip(got, want))
