"""The attention module's output written by the kernel in the projection's layout and dtype: the bits
of the fp32 per-head output cast and transposed by torch."""

import pytest
import torch

from ress_amd.aggregator import Attention, RoPE2D
from ress_amd.attention import ress_attention_forward, sparse_global_attention
from ress_amd.kernels import LayerGrid
from ress_amd.qkv import compute_qkv

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("frames", [1, 3])
def test_module_output_matches_the_cast_and_transposed_layer(dtype, frames, dev):
    torch.manual_seed(frames)
    attn = Attention(256, 4, RoPE2D()).to(dev, dtype)
    attn.proj = torch.nn.Identity()
    h, w, S = 12, 17, 5
    pos = torch.cat([torch.zeros(S, 2, dtype=torch.long),
                     torch.cartesian_prod(torch.arange(h), torch.arange(w)) + 1]).to(dev)
    pos = pos[None].repeat(2, frames, 1)
    x = torch.randn(2, frames * (S + h * w), 256, device=dev).to(dtype)
    with torch.no_grad():
        got = ress_attention_forward(attn, x, pos, num_to_select=2, num_heads=4)
        q, k, v, _ = compute_qkv(attn, x, pos, num_heads=4)
        layer = sparse_global_attention(*(t.bfloat16() for t in (q, k, v)), LayerGrid(2, 4, frames, S + h * w, S),
                                        num_to_select=2)
    want = layer.out.to(dtype).transpose(1, 2).reshape(x.shape)
    assert got.dtype == dtype and torch.equal(got, want)
