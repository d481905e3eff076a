"""The patch grid of a module call: read from the positions, or put on them by their maker."""

import pytest
import torch

from ress_amd.qkv import grid_shape


@pytest.mark.parametrize("h,w,frames,S", [(1, 1, 1, 5), (37, 37, 2, 5), (21, 37, 3, 1), (37, 21, 1, 5)])
@pytest.mark.parametrize("dtype", [torch.int64, torch.float32])
def test_grid_from_positions_and_from_their_maker(h, w, frames, S, dtype):
    pos = torch.cat([torch.zeros(S, 2), torch.cartesian_prod(torch.arange(h), torch.arange(w)).reshape(-1, 2) + 1.0])
    pos = pos.to(dtype)[None].repeat(2, frames, 1)
    x = torch.zeros(2, frames * (S + h * w), 128)
    want = {"B": 2, "N": frames, "P": S + h * w, "head_dim": 64, "num_heads": 2, "H": h, "W": w, "S": S}
    assert grid_shape(x, pos, S, 2) == want
    pos.ress_patch_grid = (h, w)
    assert grid_shape(x, pos, S, 2) == want
    pos.ress_patch_grid = (h + 1, w)  # a grid that does not fit the tokens is refused as before
    with pytest.raises(AssertionError, match="token split mismatch"):
        grid_shape(x, pos, S, 2)


def test_positions_without_a_column_are_refused():
    with pytest.raises(IndexError):
        grid_shape(torch.zeros(1, 10, 128), torch.ones(1, 10, 1), 5, 2)
