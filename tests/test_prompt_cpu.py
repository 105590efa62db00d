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
