"""The 16-bit attention's work split (csrc/attn.hip): every row of a layer against the fp32 masked
softmax, at the edges of the split's cases."""

import numpy as np
import pytest
import torch

from device_reference import row_errors
from ress_amd import kernels
from ress_amd.kernels import LayerGrid

pytestmark = pytest.mark.gpu

# (B, H, frames, P, S): rows = B * H * (ceil(frames (P-S) / 128) + ceil(frames S / 128))
CASES = [
    # one row of a full and a partial key block, whose last part is the partial block alone: the
    # waves of the upper key half see nothing but masked keys
    (1, 1, 1, 70, 5),
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
