"""decode_attention does not depend on what its workspace held: the same bytes after the allocator's blocks were filled
with NaN patterns, over unsplit and split contexts."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("NQ,NKV,hd,L", [(16, 8, 128, 200), (16, 8, 128, 1999), (2, 2, 64, 3000), (8, 1, 256, 700)])
def test_workspace_contents_do_not_matter(cuda, NQ, NKV, hd, L):
    from soinfer import ops

    g = torch.Generator(device=cuda).manual_seed(L)
    q, k, v = (torch.randn(n, generator=g, device=cuda).half() for n in (NQ * hd, NKV * L * hd, NKV * L * hd))
    args = (q.view(NQ, hd), k.view(NKV, L, hd), v.view(NKV, L, hd), L)
    want = ops.decode_attention(*args).clone()
    for _ in range(3):
        dirt = [torch.full((n,), 255, dtype=torch.uint8, device=cuda) for n in (512, 4096, 1 << 16, 1 << 18, 1 << 20)]
        del dirt
        assert torch.equal(ops.decode_attention(*args), want)
