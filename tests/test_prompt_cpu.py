"""Host-side parts of the prompt path (no GPU)."""
import pytest
import torch


def test_selection_counts_skip_entries_that_name_no_channel():
    """A token with fewer than k gates that are numbers fills its list with -1: those entries count nothing, the others
    once each, in every integer and float count type."""
    from soinfer.runtime.decoder import add_selection_counts

    sel = torch.tensor([0, 3, 4, -1, -1, -1, 3, 4, -1, -1], dtype=torch.int32)
    for dtype in (torch.int64, torch.int32, torch.float32):
        counts = torch.full((5,), 7, dtype=dtype)
        add_selection_counts(counts, sel)
        assert counts.tolist() == [8, 7, 7, 9, 9]
    counts = torch.zeros(5, dtype=torch.int64)
    add_selection_counts(counts, torch.full((6,), -1, dtype=torch.int32))
    assert int(counts.abs().sum()) == 0


# (H, I, k) -> the form measured faster than the indexed launches (None: neither is), one case on each side of every line:
# workgroups in one, two and three rounds, the bytes that go with each, the widths past 8192, 16384 and 18432 channels
FORMS = [((2048, 6144, 3072), "ordered"), ((512, 1024, 51), "ordered"), ((2560, 9728, 1945), "ordered"),
         ((2560, 9728, 4864), "ordered"), ((4096, 6144, 3993), "ordered"),
         ((4096, 12288, 1228), "ordered"), ((4096, 12288, 2457), None), ((4096, 12288, 6144), None),
         ((4096, 12288, 9830), "rows"), ((5120, 5120, 1024), "ordered"), ((5120, 5120, 1792), "rows"),
         ((5120, 5120, 4096), "rows"), ((3072, 8192, 2000), "ordered"), ((2048, 11008, 8806), "rows"),
         ((2048, 16384, 13107), "rows"), ((2048, 16384, 8192), "rows"), ((4096, 12288, 7987), "rows"),
         ((2560, 9728, 3404), None), ((5120, 17408, 3481), None),
         ((5120, 17408, 13926), None), ((1024, 20480, 1024), None)]


@pytest.mark.parametrize("shape,form", FORMS)
def test_default_dip_launches(shape, form):
    from soinfer.runtime.decoder import default_gated_form

    assert default_gated_form(*shape) == form


def config(H, I, nq, nkv, hd):
    from soinfer.runtime.decoder import DecoderConfig

    return DecoderConfig(hidden=H, layers=1, q_heads=nq, kv_heads=nkv, head_dim=hd, intermediate=I, vocab=10,
                         group_size=128, max_seq=64)


# shape, mode, k, context, tokens measured faster one at a time, tokens measured faster together
MEASURED = [((2048, 6144, 16, 8, 128), "dense", None, 0, 2, 3), ((2048, 6144, 16, 8, 128), "dense", None, 8000, 3, 4),
            ((2048, 6144, 16, 8, 128), "dense", None, 30000, 5, 8), ((1024, 3072, 8, 1, 64), "dense", None, 30000, 2, 3),
            ((256, 6144, 4, 2, 64), "dip", 1843, 0, 5, 8), ((512, 1024, 4, 2, 64), "dip", 972, 0, 3, 5),
            ((1024, 12288, 16, 8, 128), "dip", 3686, 0, 2, 3), ((1024, 12288, 16, 8, 128), "dip", 7372, 0, 3, 4),
            ((2048, 6144, 16, 8, 128), "dip", 3072, 30000, 5, 8), ((512, 1024, 4, 2, 64), "cached_dip", 614, 0, 2, 4),
            ((256, 6144, 4, 2, 64), "cached_dip", 3686, 0, 3, 5)]


@pytest.mark.parametrize("shape,mode,k,context,apart,together", MEASURED)
def test_prompt_route(shape, mode, k, context, apart, together):
    from soinfer.runtime.decoder import prompt_tokens_from

    n = prompt_tokens_from(config(*shape), mode, k, context, shape[1] // 3 if mode == "cached_dip" else None)
    assert apart < n <= together


def test_dense_prompts_on_the_matrix_cores_are_never_split_by_the_context():
    """Nine dense tokens up take one route whatever the context (their bits differ from the single steps'), and for head
    sizes up to 128 the estimate agrees."""
    from soinfer.runtime import decoder as D

    for shape in ((256, 512, 4, 2, 64), (2048, 6144, 16, 16, 128), (5120, 17408, 40, 8, 128)):
        assert D.prompt_tokens_from(config(*shape), "dense", None, 10 ** 7) <= D.PROMPT_MFMA
    # streamed weights cross the link once for all tokens together
    assert D.prompt_tokens_from(config(2048, 6144, 16, 8, 128), "dense", None, 10 ** 5, offload=True) == 3.0
