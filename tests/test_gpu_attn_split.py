"""The 16-bit attention's work split (csrc/attn.hip attn_split) at the edges of its cases: every
row of a layer against the fp32 masked softmax, for row counts on either side of each rule.
With 256 CUs (512 resident workgroups): thirds of every row up to 170 rows, the dense rows alone
up to 512, the last rows of each range beyond, in halves and thirds from 2,048 rows on."""

import numpy as np
import pytest
import torch

from device_reference import row_errors
from ress_amd import kernels
from ress_amd.kernels import LayerGrid

pytestmark = pytest.mark.gpu

# (B, H, frames, P, S): rows = B * H * (ceil(frames (P-S) / 128) + ceil(frames S / 128))
CASES = [
    (1, 1, 1, 70, 5),      # 2 rows, one key block and a partial one
    (1, 10, 1, 2053, 5),   # 170 rows: thirds of all of them
    (1, 9, 1, 2309, 5),    # 171: the dense rows alone
    (1, 9, 2, 1280, 0),    # 180 rows, no dense row: nothing split
    (1, 16, 2, 1374, 5),   # 368
    (2, 16, 3, 645, 5),    # 512: the last of the one-round launches
    (1, 27, 3, 773, 5),    # 513: the first with a tail
    (1, 23, 2, 5637, 5),   # 2,047 rows
    (1, 64, 31, 133, 5),   # 2,112 rows (two dense rows a head): halves and thirds
    (2, 64, 1, 1925, 5),   # 2,048
]


@pytest.mark.parametrize("B,H,frames,P,S", CASES)
@pytest.mark.parametrize("scale", [1.0, 8.0])  # bounded rows; running-max rows
def test_every_row_of_each_split_case(B, H, frames, P, S, scale, dev):
    grid = LayerGrid(B, H, frames, P, S)
    g = torch.Generator(device=dev).manual_seed(H * 1000 + frames)
    q, k, v = (torch.randn(B, H, grid.Tk, 64, device=dev, generator=g) for _ in range(3))
    q, k, v = (q * scale).bfloat16(), k.bfloat16(), v.bfloat16()
    keys = torch.rand(B, H, grid.q_blk_p, grid.n_cand, device=dev, generator=g)
    counts = torch.randint(0, min(grid.n_cand, 40) + 1, (B, H, grid.q_blk_p), device=dev, generator=g)
    blocks = kernels.prepare_blocks(q, k, v, grid)
    _, lut, nvalid = kernels.select_blocks(keys, counts.int(), grid, min(2, grid.n_cand))
    for dtype in (torch.float32, torch.bfloat16):
        out = kernels.sparse_attention(blocks, lut, nvalid, out_dtype=dtype)
        err, cos = row_errors(out, q, k, v, grid, lut, nvalid)
        assert not np.isnan(err).any()
        # the attention's bar, and half an ulp of the output's own rounding (2^-9 of its magnitude)
        bound = 2e-2 + (2**-9 * out.abs().max().item() if dtype == torch.bfloat16 else 0.0)
        assert err.max() < bound, (err.max(), np.unravel_index(err.argmax(), err.shape))
        assert cos.min() > 0.999
