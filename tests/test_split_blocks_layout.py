"""Row blocks of a weight that is not contiguous are refused as the weight itself is, also where a block alone would pass."""
import pytest
import torch

from dion_amd.optimizers import _row_blocks


def test_row_blocks():
    w = torch.arange(24.0).view(4, 6)
    assert [b.tolist() for b in _row_blocks([w], (1, [0, 3]))] == [[w[0].tolist()], [w[3].tolist()]]
    for view in (w[:, :5], w.T):
        with pytest.raises(ValueError, match="contiguous"):
            _row_blocks([view], (1, [0, 1]))
