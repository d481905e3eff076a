"""The budget kernels at the edges of their walks, bit for bit against the oracle: head counts around
the reallocation's lane bounds."""

import numpy as np
import pytest
import torch

import oracle
from ress_amd import budget, kernels, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H", [1, 4, 8, 9, 16, 17, 24, 32, 33, 64])
@pytest.mark.parametrize("B,q_blk,beta", [(1, 1, 1.0), (2, 5, 1.0), (3, 43, 0.5)])
def test_head_budget_head_counts(H, B, q_blk, beta, dev):
    rng = np.random.default_rng(H)
    base = rng.integers(0, 342, size=(B, H, q_blk)).astype(np.int32)
    base[0, 0] = 341
    scores = torch.from_numpy(np.exp(rng.normal(size=H)).astype(np.float32))
    norm = torch.from_numpy(budget.scores_norm(scores)).to(dev)
    iters = torch.empty(B, q_blk, dtype=torch.int32, device=dev)
    got = kernels.head_budget(torch.from_numpy(base).to(dev), norm, beta, 342, min_select=2, iters_out=iters)
    # the reallocation is column by column, so a batch entry is a call of its own
    for b in range(B):
        want, it = oracle.head_budget(base[b:b + 1], oracle.scores_norm_seq(scores.numpy()), beta, 342, min_select=2)
        assert np.array_equal(got[b:b + 1].cpu().numpy(), want)
        assert iters[b].max().item() == it
    uniform = kernels.head_budget(torch.from_numpy(base).to(dev), None, beta, 342, min_select=2, iters_out=iters)
    assert np.array_equal(uniform.cpu().numpy(), np.maximum(base, 2)) and not iters.any()
