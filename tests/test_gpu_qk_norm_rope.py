"""The fused q/k-norm + RoPE kernel at the edges of its walk: token counts around the workgroup's
eight, head counts that fill its 32-head steps partly and over several, batches, buffers that are
only 8-byte aligned, no positions, and positions past the hardware sine's range."""

import pytest
import torch

from ress_amd import _lib
from ress_amd.aggregator import RoPE2D

pytestmark = pytest.mark.gpu


def _call(qkv, B, T, nh, w, pos, out):
    P = _lib.ptr
    _lib.call("ress_qk_norm_rope", P(qkv), B, T, nh, P(w[0]), P(w[1]), P(w[2]), P(w[3]), 1e-5, P(pos), 100.0,
              *(P(o) for o in out), _lib.stream_handle(qkv.device))
    return out


@pytest.mark.parametrize("B,T,nh", [(1, 1, 1), (2, 7, 3), (1, 8, 16), (3, 9, 24), (1, 37, 64), (2, 1374, 16)])
@pytest.mark.parametrize("max_pos", [0, 38, 5000])
def test_against_float64_and_across_alignments(B, T, nh, max_pos, dev):
    g = torch.Generator(device=dev).manual_seed(T * nh)
    n = B * T * 3 * nh * 64
    store = torch.randn(n + 8, device=dev, generator=g).bfloat16()
    qkv = store[:n].view(B, T, 3, nh, 64)
    w = [(torch.randn(64, device=dev, generator=g) * 0.2 + (1 - i % 2)).bfloat16() for i in range(4)]
    pos = torch.randint(0, max_pos, (B, T, 2), device=dev, generator=g) if max_pos else None
    out = _call(qkv, B, T, nh, w, pos, [torch.empty(B, nh, T, 64, dtype=torch.bfloat16, device=dev) for _ in range(3)])
    # the same values from buffers 8 bytes past a 16-byte boundary
    off = store.clone()
    off[4:n + 4] = store[:n]
    bufs = [torch.empty(B * nh * T * 64 + 4, dtype=torch.bfloat16, device=dev)[4:].view(B, nh, T, 64) for _ in range(3)]
    got8 = _call(off[4:n + 4], B, T, nh, w, pos, bufs)
    for a, b in zip(out, got8):
        assert torch.equal(a.view(torch.int16), b.view(torch.int16))
    q, k, v = qkv.permute(2, 0, 3, 1, 4)
    assert torch.equal(out[2].view(torch.int16), v.contiguous().view(torch.int16))
    for got, x, gain, bias in ((out[0], q, w[0], w[1]), (out[1], k, w[2], w[3])):
        y = torch.nn.functional.layer_norm(x.double(), (64,), gain.double(), bias.double(), 1e-5)
        if pos is not None:
            inv = 100.0 ** (-torch.arange(0, 32, 2, device=dev, dtype=torch.float64) / 32)
            parts = []
            for axis in (0, 1):
                a, b = y[..., 32 * axis:32 * axis + 16], y[..., 32 * axis + 16:32 * axis + 32]
                ang = pos[:, None, :, axis, None].double() * inv
                parts += [a * ang.cos() - b * ang.sin(), b * ang.cos() + a * ang.sin()]
            y = torch.cat(parts, dim=-1)
        # two bf16 roundings (2^-9 of the norm's and of the rotation's value, |y| below 8 here), and
        # the fp32 angle's: 2^-24 of at most 5,000 rad
        assert (got.double() - y).abs().max().item() <= 8 * (2**-9 + 2**-8) + 8 * max_pos * 2**-23


def test_the_module_rotation_is_the_kernels(dev):
    """RoPE2D (the torch module) and the kernel on normalised inputs of unit gain."""
    B, T, nh = 1, 50, 4
    g = torch.Generator(device=dev).manual_seed(1)
    qkv = torch.randn(B, T, 3, nh, 64, device=dev, generator=g).bfloat16()
    one, zero = torch.ones(64, device=dev).bfloat16(), torch.zeros(64, device=dev).bfloat16()
    pos = torch.randint(0, 38, (B, T, 2), device=dev, generator=g)
    out = _call(qkv, B, T, nh, [one, zero, one, zero], pos,
                [torch.empty(B, nh, T, 64, dtype=torch.bfloat16, device=dev) for _ in range(3)])
    y = torch.nn.functional.layer_norm(qkv[:, :, 0].transpose(1, 2).float(), (64,)).bfloat16()
    assert (out[0].float() - RoPE2D()(y, pos).float()).abs().max().item() <= 8 * 2**-8
