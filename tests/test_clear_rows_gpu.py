"""A request's rows of all state tensors cleared in one launch."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("widths", [[16], [1, 3], [4, 8, 1031], [70001, 5, 65536, 12]])
@pytest.mark.parametrize("dtype", [torch.uint8, torch.bfloat16, torch.float32, torch.float64])
def test_one_row_of_every_tensor(widths, dtype):
    """Rows of 16 bytes and their remainders, of one element, and of more than a block's stores; the rows beside stay."""
    from mlx_lm_amd.ops import kernels

    other = torch.float32 if dtype == torch.uint8 else torch.uint8
    tensors = [torch.full((5, w), 7, dtype=dtype if i % 2 == 0 else other, device="cuda") for i, w in enumerate(widths)]
    rows = kernels.RowsCleared(tensors)
    for row in (0, 4, 2):
        rows.clear(row)
    for t in tensors:
        assert not t[[0, 2, 4]].any() and (t[[1, 3]] == 7).all()
    for row in (-1, 5):
        with pytest.raises(Exception):
            rows.clear(row)
