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


@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
@pytest.mark.parametrize("token", [5, 21, 70, 1373])
def test_a_query_that_is_not_finite_leaves_the_others_alone(bad, token, dev):
    """The queries of a row share MFMAs: one with NaN or infinity may spoil its own output only.
    The clean run's rows are running-max rows too, so the outputs' numerators keep their bits; the
    row sum of such a row is formed in another order, of n positive fp32 terms: two orders differ by
    2 n 2^-24 of the sum at most."""
    grid = LayerGrid(1, 2, 1, 1374, 5)
    g = torch.Generator(device=dev).manual_seed(token)
    q, k, v = (torch.randn(1, 2, grid.Tk, 64, device=dev, generator=g) for _ in range(3))
    q, k, v = (q * 8).bfloat16(), k.bfloat16(), v.bfloat16()
    blocks = kernels.prepare_blocks(q, k, v, grid)
    lut = torch.arange(grid.kb_tot, dtype=torch.int32, device=dev).expand(2, grid.q_blk_total, -1).contiguous()
    nvalid = torch.full((2, grid.q_blk_total), grid.kb_tot, dtype=torch.int32, device=dev)
    clean = kernels.sparse_attention(blocks, lut, nvalid, out_dtype=torch.float32).clone()
    q[0, 1, token, 3] = bad
    out = kernels.sparse_attention(kernels.prepare_blocks(q, k, v, grid), lut, nvalid, out_dtype=torch.float32)
    assert torch.isnan(out[0, 1, token]).all()
    out[0, 1, token] = clean[0, 1, token]
    assert ((out - clean).abs() <= 2 * grid.kb_tot * 64 * 2**-24 * clean.abs()).all()
    out[0, 1, :], clean[0, 1, :] = 0, 0
    assert torch.equal(out, clean)  # the other head's rows: the same bits


@pytest.mark.parametrize("bad", [float("nan"), -float("nan"), float("inf"), -float("inf"), 7e4, 6.2e4])
@pytest.mark.parametrize("scale", [1.0, 8.0])  # the other queries alone: a bounded row; a running-max row
@pytest.mark.parametrize("keys", [1.0, 0.0])   # zero keys: every bound is 0 times the query's norm
def test_a_rows_path_does_not_hang_on_one_query(bad, scale, keys, dev):
    """NaN of either sign, infinity, a value past fp16 and one just inside it: the other queries of its
    row, and of every row, keep to the attention's bar; a value fp16 holds keeps its own output too."""
    grid = LayerGrid(1, 2, 1, 1374, 5)
    g = torch.Generator(device=dev).manual_seed(7)
    q, k, v = (torch.randn(1, 2, grid.Tk, 64, device=dev, generator=g) for _ in range(3))
    q, k, v = (q * scale).bfloat16(), (k * keys).bfloat16(), v.bfloat16()
    q[0, 1, 300, 9] = bad
    lut = torch.arange(grid.kb_tot, dtype=torch.int32, device=dev).expand(2, grid.q_blk_total, -1).contiguous()
    nvalid = torch.full((2, grid.q_blk_total), grid.kb_tot, dtype=torch.int32, device=dev)
    out = kernels.sparse_attention(kernels.prepare_blocks(q, k, v, grid), lut, nvalid, out_dtype=torch.float32)
    fits = abs(bad) < 65520.0  # False for NaN
    assert out.ress_attn_status.item() == (0 if fits else 2)
    ref = torch.softmax(torch.matmul(q.float(), k.float().transpose(-1, -2).contiguous()) / 8, dim=-1) @ v.float()
    err = (out - ref).abs().amax(-1)
    if not fits:
        err[0, 1, 300] = 0.0
    assert not torch.isnan(err).any() and err.max().item() < 2e-2
