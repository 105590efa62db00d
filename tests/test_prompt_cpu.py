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
         ((2048, 16384, 13107), "rows"), ((2048, 16384, 8192), "rows"), ((4096, 12288, 7987), "rows"), ((2560, 9728, 3404), None), ((5120, 17408, 3481), None),
         ((5120, 17408, 13926), None), ((1024, 20480, 1024), None)]


@pytest.mark.parametrize("shape,form", FORMS)
def test_default_dip_launches(shape, form):
    from soinfer.runtime.decoder import default_gated_form

    assert default_gated_form(*shape) == form
