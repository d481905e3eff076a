"""The Q/K/V block passes, a workgroup of four waves per block, bit for bit against the oracle where
their rows, waves and tiles end: blocks of one row, of a row past a wave's eight or a pass's 32, with
and without special tokens, the pools over the patch keys or every key, permuted tokens, strided inputs."""

import numpy as np
import pytest
import torch

import oracle
from ress_amd import kernels
from ress_amd.kernels import LayerGrid

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("frames,P,S", [
    (1, 1, 0), (1, 8, 0), (1, 9, 1), (1, 33, 0), (1, 64, 0), (1, 65, 0), (1, 128, 0), (1, 129, 0), (2, 97, 33),
    (3, 70, 5), (5, 63, 31), (2, 161, 1)])
@pytest.mark.parametrize("mode", ["f16", "i8", "i8x2"])
@pytest.mark.parametrize("pool_all", [False, True])
@pytest.mark.parametrize("form", ["plain", "strided", "permuted"])
def test_block_passes_match_the_oracle(frames, P, S, mode, pool_all, form, dev):
    B, H, N = 2, 3, frames * P
    gen = torch.Generator().manual_seed(N)
    q, k, v = (torch.randn(B, H, N, 64, generator=gen).bfloat16() for _ in range(3))
    k[0, 0, N // 2, 5] = 7e4      # beyond fp16: an infinite norm
    k[1, 1, N - 1] = 0.0          # a zero row; in the smallest grid a zero block, whose scale is 0
    v[1, 2, :, 7] = -0.0
    q[0, 1, 0, 9] = -300.0
    tq, tk, tv, order = q, k, v, None
    if form == "permuted":
        perm = torch.randperm(P - S, generator=gen)
        order = perm.to(torch.int32).to(dev)
        at = torch.cat([torch.cat([torch.arange(S), S + perm]) + f * P for f in range(frames)])
        q, k, v = (x[:, :, at] for x in (q, k, v))  # the oracle takes the tokens in block order
    if form == "strided":  # one projection's (B, N, 3, H, 64)
        tq, tk, tv = torch.stack([x.transpose(1, 2) for x in (tq, tk, tv)], dim=2).to(dev).transpose(1, 3).unbind(2)
    g = LayerGrid(B, H, frames, P, S, sink_mass=pool_all)
    blocks = kernels.prepare_blocks(tq.to(dev), tk.to(dev), tv.to(dev), g, mode=mode, patch_order=order)
    o = oracle.prep_qkv(q, k, v, frames, P, S, pool_all=pool_all)
    fields = ["pooled_q", "pooled_k", "pooled_v", "v_pack"]
    if mode != "f16":
        fields += ["q_i8", "q_scale", "k_i8", "k_scale", "ksum", "km"] + (["q_lo", "k_lo"] if mode == "i8x2" else [])
    for f in fields:
        got = getattr(blocks, f).cpu()
        got = got.view(torch.int16) if got.dtype == torch.bfloat16 else got
        assert got.numpy().tobytes() == o[f].tobytes(), f
    if mode == "f16":
        assert blocks.k_scale.cpu().numpy().tobytes() == o["k_norm"].tobytes()
        T = S * frames
        keys = torch.cat([k.view(B, H, frames, P, 64)[..., S:, :].reshape(B, H, N - T, 64),
                          k.view(B, H, frames, P, 64)[..., :S, :].reshape(B, H, T, 64)], dim=2)
        want = torch.zeros(B * H, g.kb_tot * 64, 64, dtype=torch.float16)
        want[:, :N] = keys.reshape(B * H, N, 64).to(torch.float16)
        assert torch.equal(blocks.k_pack.cpu().view_as(want), want)
