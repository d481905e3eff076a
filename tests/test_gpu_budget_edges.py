"""The budget kernels at the edges of their walks, bit for bit against the oracle: row lengths around
the CDF sort's powers of two, its register form's limit of 2,048 and the prefix chain's batches;
head counts around the reallocation's lane bounds."""

import numpy as np
import pytest
import torch

import oracle
from ress_amd import budget, kernels, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 31, 32, 33, 127, 128, 129, 255, 256, 257, 342, 512, 513, 1024, 1025, 2047, 2048, 2049, 4293])
@pytest.mark.parametrize("sr,cdf", [(None, 0.9), (0.5, 0.7), (0.95, 0.999), (None, 2.0)])
def test_cdf_count_row_lengths(n, sr, cdf, dev):
    rng = np.random.default_rng(n)
    a = rng.dirichlet(np.full(n, 0.3), size=(1, 2, 7)).astype(np.float32)
    a[0, 0, 0] = np.float32(1 / n)      # ties everywhere
    a[0, 0, 1] = 0.0                    # never crosses
    a[0, 0, 2, :] = 0.0
    a[0, 0, 2, n // 2] = 1.0            # crosses at once, or (cdf 2) never
    got = budget.compute_baseline_num_to_select(torch.from_numpy(a).to(dev), sr, cdf)
    assert np.array_equal(got.cpu().numpy(), oracle.baseline_budget(a, sr, cdf))
    # a score map, whose prefix sums rise and fall again: the count up to the first one past the cut
    raw = rng.normal(size=n).astype(np.float32)
    c, thr, first = np.float32(0), np.float32(np.float32(cdf) + np.float32(1e-5)), n
    for i, x in enumerate(np.sort(raw)[::-1]):
        c = np.float32(c + x)
        if c > thr:
            first = i
            break
    got = budget.compute_baseline_num_to_select(torch.from_numpy(raw)[None].to(dev), sr, cdf)
    assert got.item() == max(first, int(n * (1 - sr)) if sr is not None else 0)


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
