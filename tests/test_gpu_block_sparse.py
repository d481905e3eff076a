"""run_block_sparse_kernel's folded casts and the key-mean pass against the SpargeAttn mirror's own
call sequence and the K/V block pass: the same operations in the same order, so the same bits."""

import numpy as np
import pytest
import torch

from ress_amd import _lib, sparge
from ress_amd.attention import run_block_sparse_kernel

pytestmark = pytest.mark.gpu


def _inputs(B, H, Tq, Tk, v_dtype, dev):
    g = torch.Generator(device=dev).manual_seed(Tq + Tk)
    q, k, v = (torch.randn(B, H, T, 64, device=dev, generator=g) for T in (Tq, Tk, Tk))
    v[..., 3] *= 3e4  # bf16 values past fp16's range among them
    fmap = torch.rand(B, H, -(-Tq // 128), -(-Tk // 64), device=dev, generator=g) < 0.4
    fmap[:, :, 0] = False  # a row that keeps nothing
    return q.bfloat16(), k.bfloat16(), v.to(v_dtype), fmap


@pytest.mark.parametrize("Tq,Tk", [(1, 1), (128, 64), (129, 65), (260, 330), (1000, 4161)])
@pytest.mark.parametrize("v_dtype,dtype,out_dtype", [
    (torch.bfloat16, torch.float16, torch.float32), (torch.bfloat16, torch.bfloat16, torch.float32),
    (torch.float32, torch.float16, torch.float32), (torch.float16, torch.float16, torch.float16),
    (torch.bfloat16, torch.float16, torch.bfloat16), (torch.bfloat16, torch.float32, torch.float32)])
def test_folded_casts_match_the_mirror(Tq, Tk, v_dtype, dtype, out_dtype, dev):
    B, H = 2, 3
    q, k, v, fmap = _inputs(B, H, Tq, Tk, v_dtype, dev)
    got, sparsity = run_block_sparse_kernel(q, k, v, fmap, dtype=dtype, out_dtype=out_dtype)
    half = dtype in (torch.float16, torch.bfloat16)
    q8, qs, k8, ks = sparge.per_block_int8(q, k, km=sparge.key_mean(k))
    lut, nv = sparge.block_map_lut_triton(fmap.to(torch.uint8))
    o = torch.empty(B, H, Tq, 64, dtype=dtype if half else out_dtype, device=dev)
    sparge.qk_int8_sv_f16_accum_f16_block_sparse_attn_inst_buf_with_pv_threshold(
        q8, k8, v.to(dtype), o, lut, nv, sparge.hyperparameter_check(1e10, H, dev), qs, ks, 1, 0, 1, 0.125, 0)
    sparge.check_last_call()
    want = o.to(out_dtype)
    assert got.dtype == out_dtype
    assert torch.equal(torch.isnan(got), torch.isnan(want))
    assert torch.equal(got.nan_to_num(), want.nan_to_num())
    assert sparsity == pytest.approx(1 - fmap.double().mean().item(), abs=1e-12)


@pytest.mark.parametrize("H,nq", [(12, 25), (16, 50), (21, 100)])  # no row split; the last rows in thirds; halves too
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_rounded_fp32_output_of_each_split(H, nq, dtype, dev):
    """300, 800 and 2,100 rows: whole rows stored by the attention kernel, parts by the merge."""
    q, k, v, fmap = _inputs(1, H, 128 * nq - 37, 330, torch.bfloat16, dev)
    got, _ = run_block_sparse_kernel(q, k, v, fmap, dtype=dtype)
    q8, qs, k8, ks = sparge.per_block_int8(q, k, km=sparge.key_mean(k))
    lut, nv = sparge.block_map_lut_triton(fmap)
    o = torch.empty(q.shape, dtype=dtype, device=dev)
    sparge.qk_int8_sv_f16_accum_f16_block_sparse_attn_inst_buf_with_pv_threshold(
        q8, k8, v.to(dtype), o, lut, nv, sparge.hyperparameter_check(1e10, H, dev), qs, ks, 1, 0, 1, 0.125, 0)
    assert got.dtype == torch.float32
    assert torch.equal(got.nan_to_num(), o.float().nan_to_num()) and torch.equal(got.isnan(), o.isnan())


@pytest.mark.parametrize("off", [1, 4])  # elements past a 16-byte boundary
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_a_value_that_is_not_16_byte_aligned(off, dtype, dev):
    """A contiguous bf16 V at any storage offset, where P V runs in fp16: the aligned V's bits."""
    q, k, v, fmap = _inputs(2, 3, 260, 330, torch.bfloat16, dev)
    store = torch.empty(v.numel() + off, dtype=torch.bfloat16, device=dev)
    shifted = store[off:].view(v.shape)
    shifted.copy_(v)
    assert shifted.is_contiguous() and shifted.data_ptr() % 16
    got, _ = run_block_sparse_kernel(q, k, shifted, fmap, dtype=dtype)
    want, _ = run_block_sparse_kernel(q, k, v, fmap, dtype=dtype)
    assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(got.nan_to_num(), want.nan_to_num())


@pytest.mark.parametrize("Tq,nk", [(32, 1), (32, 7), (128 * 60, 9)])  # parts of one block, of several, whole rows too
@pytest.mark.parametrize("v_dtype", [torch.float16, torch.bfloat16])
def test_a_query_whose_scores_overflow_leaves_the_others_alone(Tq, nk, v_dtype, dev):
    """Query 3 of each 32 meets every key of block 0 (and of the last) with a score far below fp32's
    range; the others score 0 everywhere, so their output is the mean of V over the keys."""
    B, H, Tk = 1, 16, 64 * nk
    g = torch.Generator(device=dev).manual_seed(nk)
    q8 = torch.zeros(B, H, Tq, 64, dtype=torch.int8, device=dev)
    q8[:, :, 3::32] = -100
    k8 = torch.zeros(B, H, Tk, 64, dtype=torch.int8, device=dev)
    k8[:, :, :64], k8[:, :, -64:] = 100, 100
    v = torch.randn(B, H, Tk, 64, device=dev, generator=g).to(v_dtype)
    nq = -(-Tq // 128)
    qs = torch.full((B, H, nq), 1e20, device=dev)
    ks = torch.full((B, H, nk), 1e15, device=dev)  # scores of -640,000 * 1e35 / 8
    lut = torch.arange(nk, dtype=torch.int32, device=dev).expand(B, H, nq, nk).contiguous()
    nv = torch.full((B, H, nq), nk, dtype=torch.int32, device=dev)
    o = torch.empty(B, H, Tq, 64, device=dev)
    sparge.qk_int8_sv_f16_accum_f16_block_sparse_attn_inst_buf_with_pv_threshold(
        q8, k8, v, o, lut, nv, sparge.hyperparameter_check(1e10, H, dev), qs, ks, 1, 0, 1, 0.125, 0)
    sparge.check_last_call()
    others = torch.arange(Tq, device=dev) % 32 != 3
    want = v.float().mean(2, keepdim=True)
    # fp32 sums of Tk terms below 5 and a division: 2 Tk 2^-24 of the largest term
    assert ((o[:, :, others] - want).abs() <= 2 * Tk * 2**-24 * 5).all()


def test_a_map_of_another_shape_is_refused(dev):
    q, k, v, fmap = _inputs(1, 2, 260, 330, torch.bfloat16, dev)
    with pytest.raises(ValueError, match="lut must be"):
        run_block_sparse_kernel(q, k, v, fmap[..., :-1])
    with pytest.raises(ValueError, match="lut must be"):  # too few heads
        run_block_sparse_kernel(q, k, v, fmap[:, :1])


def test_a_map_with_batch_and_heads_in_one_dim(dev):
    q, k, v, fmap = _inputs(2, 3, 260, 330, torch.float16, dev)
    want, sparsity = run_block_sparse_kernel(q, k, v, fmap)
    for lead in ((1, 6), (6, 1)):
        got, s = run_block_sparse_kernel(q, k, v, fmap.view(*lead, *fmap.shape[2:]))
        assert torch.equal(got.nan_to_num(), want.nan_to_num()) and s == sparsity


def test_the_last_calls_status_after_a_bad_mirror_call(dev):
    q, k, v, fmap = _inputs(1, 2, 260, 330, torch.float16, dev)
    q8, qs, k8, ks = sparge.per_block_int8(q, k)
    lut, nv = sparge.block_map_lut_triton(fmap)
    sparge.qk_int8_sv_f16_accum_f16_block_sparse_attn_inst_buf_with_pv_threshold(
        q8, k8, v, torch.empty_like(v[:, :, :260]), lut, nv, sparge.hyperparameter_check(5.0, 2, dev), qs, ks, 1, 0, 1,
        0.125, 0)  # a PV threshold is not provided: the status word says so
    assert sparge.last_call_status().tolist() == [4]
    run_block_sparse_kernel(q, k, v, fmap)
    status = sparge.last_call_status()
    assert status.device == dev and status.dtype == torch.int32 and status.tolist() == [0]
    sparge.check_last_call()


@pytest.mark.parametrize("Tk", [1, 63, 64, 65, 4096, 4097, 8200])  # up to 64 blocks, 65, two chunks and a bit
@pytest.mark.parametrize("strided", [False, True])
def test_key_mean_matches_the_block_pass(Tk, strided, dev):
    B, H = 2, 3
    g = torch.Generator(device=dev).manual_seed(Tk)
    k = torch.randn(B, Tk, H, 64, device=dev, generator=g).bfloat16().transpose(1, 2)
    k = k if strided else k.contiguous()
    nk = -(-Tk // 64)
    ksum, pk, pv = (torch.empty(B * H, nk, 64, device=dev) for _ in range(3))
    km = torch.empty(B * H, 64, device=dev)
    vp = torch.empty(B * H, nk, 4096, dtype=torch.bfloat16, device=dev)
    _lib.call("ress_prep_kv_plain", _lib.ptr(k), _lib.ptr(k), B, H, Tk, *k.stride()[:3], *k.stride()[:3],
              _lib.ptr(ksum), _lib.ptr(km), _lib.ptr(pk), _lib.ptr(pv), _lib.ptr(vp), _lib.stream_handle(dev))
    assert torch.equal(sparge.key_mean(k), km)
    # the sums' order: blocks in sequence, in fp32, then one IEEE division (torch's division by a
    # number multiplies by its reciprocal)
    acc, sums = np.zeros((B * H, 64), np.float32), ksum.cpu().numpy()
    for b in range(nk):
        acc = acc + sums[:, b]
    assert np.array_equal(km.cpu().numpy(), acc / np.float32(Tk))
