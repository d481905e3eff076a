"""The attention's work split (csrc/attn.hip attn_split) at the edges of its cases: every row of a
layer against the fp32 masked softmax, for row counts on either side of each rule. With 256 CUs and
512 resident workgroups of the 16-bit kernel (768 of the INT8 kernel): thirds of every row up to 170
rows (256), the dense rows alone up to 512 (768), the last rows of each range beyond, in halves and
thirds from 2,048 rows on."""

import numpy as np
import pytest
import torch

from device_reference import RESIDENT, attn_schedule, kernel_order, row_errors
from ress_amd import _lib, kernels
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
INT8_CASES = [
    (1, 1, 1, 70, 5),      # 2 rows
    (1, 16, 1, 1925, 5),   # 256: thirds of all of them
    (1, 6, 1, 5381, 5),    # 258: the dense rows alone
    (1, 9, 4, 1280, 0),    # 360 rows, no dense row: nothing split
    (1, 16, 1, 6021, 5),   # 768: the last of the one-round launches
    (1, 22, 1, 4357, 5),   # 770: a tail
    (1, 23, 2, 5637, 5),   # 2,047 rows
    (2, 64, 1, 1925, 5),   # 2,048: halves and thirds
]


def _layer(B, H, frames, P, S, scale, mode, dev):
    """q, k, v, the prepared blocks, LUT and counts of a layer that keeps up to 40 random blocks a row."""
    grid = LayerGrid(B, H, frames, P, S)
    g = torch.Generator(device=dev).manual_seed(H * 1000 + frames)
    q, k, v = (torch.randn(B, H, grid.Tk, 64, device=dev, generator=g) for _ in range(3))
    q, k, v = (q * scale).bfloat16(), k.bfloat16(), v.bfloat16()
    keys = torch.rand(B, H, grid.q_blk_p, grid.n_cand, device=dev, generator=g)
    counts = torch.randint(0, min(grid.n_cand, 40) + 1, (B, H, grid.q_blk_p), device=dev, generator=g)
    blocks = kernels.prepare_blocks(q, k, v, grid, mode=mode)
    _, lut, nvalid = kernels.select_blocks(keys, counts.int(), grid, min(2, grid.n_cand))
    return grid, q, k, v, blocks, lut, nvalid


@pytest.mark.parametrize("B,H,frames,P,S", CASES)
@pytest.mark.parametrize("scale", [1.0, 8.0])  # bounded rows; running-max rows
def test_every_row_of_each_split_case(B, H, frames, P, S, scale, dev):
    grid, q, k, v, blocks, lut, nvalid = _layer(B, H, frames, P, S, scale, "f16", dev)
    for dtype in (torch.float32, torch.bfloat16):
        out = kernels.sparse_attention(blocks, lut, nvalid, out_dtype=dtype)
        err, cos = row_errors(out, q, k, v, grid, lut, nvalid)
        assert not np.isnan(err).any()
        # the attention's bar, and half an ulp of the output's own rounding (2^-9 of its magnitude)
        bound = 2e-2 + (2**-9 * out.abs().max().item() if dtype == torch.bfloat16 else 0.0)
        assert err.max() < bound, (err.max(), np.unravel_index(err.argmax(), err.shape))
        assert cos.min() > 0.999


def _decoded(hi, lo, scale, tokens):
    """fp32 (BH, tokens, 64) of INT8 codes [BH][blocks][rows][64] with one scale per block."""
    x = hi.float() if lo is None else hi.float() + lo.float() / 254
    return (x * scale[..., None, None]).flatten(1, 2)[:, :tokens]


@pytest.mark.parametrize("B,H,frames,P,S", INT8_CASES)
@pytest.mark.parametrize("mode", ["i8", "i8x2"])
def test_every_row_of_each_split_case_int8(B, H, frames, P, S, mode, dev):
    """Against the softmax over the values that the codes stand for (the keys' mean, which the codes
    leave out, moves all scores of a query alike), so that both modes meet the attention's bar."""
    grid, q, k, v, blocks, lut, nvalid = _layer(B, H, frames, P, S, 1.0, mode, dev)
    qd, kd = torch.empty(B, H, grid.Tk, 64, device=dev), torch.empty(B, H, grid.Tk, 64, device=dev)
    order = kernel_order(frames, P, S, dev)
    rows = torch.cat([_decoded(blocks.q_i8[:, s], None if blocks.q_lo is None else blocks.q_lo[:, s], blocks.q_scale[:, s], n)
                      for s, n in ((slice(grid.q_blk_p), grid.T_p), (slice(grid.q_blk_p, None), grid.T_s))], dim=1)
    qd[:, :, order] = rows.view(B, H, -1, 64)
    kd[:, :, order] = _decoded(blocks.k_i8, blocks.k_lo, blocks.k_scale, grid.Tk).view(B, H, -1, 64)
    for dtype in (torch.float32, torch.bfloat16):
        out = kernels.sparse_attention(blocks, lut, nvalid, out_dtype=dtype)
        err, cos = row_errors(out, qd, kd, v, grid, lut, nvalid)
        assert not np.isnan(err).any()
        bound = 2e-2 + (2**-9 * out.abs().max().item() if dtype == torch.bfloat16 else 0.0)
        assert err.max() < bound, (err.max(), np.unravel_index(err.argmax(), err.shape))
        assert cos.min() > 0.999


CHUNKED = (1, 64, 1, 32837, 5)  # 514 key blocks a head, 514 MiB of K/V: rows chunk-major


@pytest.mark.parametrize("mode,case", [("f16", c) for c in CASES + [CHUNKED]]
                         + [(m, c) for c in INT8_CASES for m in ("i8", "i8x2")])
def test_the_split_restated(mode, case, dev):
    """device_reference.attn_schedule, by which other tests name the split rows, against a launch: its
    ranges, and as many part slots written as it counts parts of split rows."""
    grid, q, k, v, blocks, lut, nvalid = _layer(*case, 1.0, mode, dev)
    n = _lib.lib().ress_attn_sched_bytes(grid.B, grid.H, grid.Tk)
    sched = torch.full((n,), 0xFF, dtype=torch.uint8, device=dev)
    out, P = torch.empty(grid.B, grid.H, grid.Tk, 64, device=dev), _lib.ptr
    tail = (P(lut), P(nvalid), grid.B, grid.H, grid.frames, grid.P, grid.S, None, 0.125, P(out), 0, *out.stride()[:3],
            P(sched), _lib.stream_handle(dev))
    if mode == "f16":
        _lib.call("ress_sparse_attn_fwd_f16", P(q), *q.stride()[:3], P(blocks.k_pack), P(blocks.k_scale), P(blocks.v_pack), *tail)
    else:
        _lib.call("ress_sparse_attn_fwd", P(blocks.q_i8), P(blocks.q_lo), P(blocks.q_scale), P(blocks.k_i8), P(blocks.k_lo),
                  P(blocks.k_scale), P(blocks.v_pack), 0, *tail)
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    parts, bounds = attn_schedule(nvalid.cpu().numpy(), grid.q_blk_p, grid.kb_tot, mode, cus)
    assert sched[:36].view(torch.int32).tolist() == bounds
    slot = 4 * (256 * 32 + 2 * 256)
    written = (sched[256:].view(-1, slot) != 0xFF).any(1).sum().item()
    assert written == parts[parts > 1].sum()
    if parts.size > RESIDENT[mode] * cus:
        assert (parts > 1).sum() == sum(min(b - a, 40 if parts.size >= 8 * cus else 32) for a, b in zip(bounds, bounds[1:]))


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
