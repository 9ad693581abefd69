"""The Sparse-Q queries and forced tokens of a gap mask: one call against the
mask functions on torch, for every form of mask and tail."""

import numpy as np
import pytest
import torch

from cacheblend_vllm import selection as S
from cacheblend_vllm.config import CacheBlendConfig

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)


# token counts around the 8-token groups and 2048-token tiles, many tiles
@pytest.mark.parametrize("n", [1, 7, 8, 9, 2047, 2048, 2049, 6001, 70000])
@pytest.mark.parametrize("radius", [0, 1, 16, 4096])
def test_rows_match_the_mask_functions(n, radius):
    g = torch.Generator().manual_seed(n)
    sparse = torch.rand(n, generator=g) < 0.01
    masks = [torch.zeros(n, dtype=torch.bool), torch.ones(n, dtype=torch.bool), sparse,
             torch.arange(n) == n - 1, torch.arange(n) == 0]
    wide = torch.zeros(n + 3, dtype=torch.bool)
    wide[3:] = sparse
    strided = torch.zeros(n, 2, dtype=torch.bool)
    strided[:, 1] = sparse
    devs = [m.to(DEV) for m in masks] + [wide.to(DEV)[3:], strided.to(DEV)[:, 1]]
    for i, gap in enumerate(devs):
        for tail in (0, 1, 64, n, n + 5):
            print(f"n={n} radius={radius} mask {i} tail={tail}", flush=True)
            count = int(gap.sum())
            query, forced, has_gap = S.sparse_q_masks(gap, tail, radius, gap_count=count)
            want = S.sparse_q_query_rows(query, has_gap, count, tail)
            rows, got, got_count = S.sparse_q_rows(gap, tail, radius)
            assert got_count == count
            assert torch.equal(rows, want)
            assert torch.equal(got, forced)


@pytest.mark.parametrize("block", [16, np.int64(16), 16.0])
@pytest.mark.parametrize("tail", [64, np.int64(64)])
def test_sizes_of_any_whole_number_type(block, tail):
    n, g = 300, torch.Generator().manual_seed(5)
    q, k = torch.randn(n, 2, 64, generator=g).to(DEV), torch.randn(n, 1, 64, generator=g).to(DEV)
    index = torch.arange(n, device=DEV)
    config = CacheBlendConfig.from_extra_config({"selection_strategy": "sparse_q", "tail_query_tokens": tail})
    for gap in (torch.zeros(n, dtype=torch.bool), torch.arange(n) == 100):
        want_q, want, _ = S.sparse_q_masks(gap.to(DEV), 64, 16)
        _, forced, stats = S.BlendSelector(config, block)._sparse_q_scores(q, k, index, gap.to(DEV), 0.125)
        assert torch.equal(forced, want) and stats["sparse_query_tokens"] == int(want_q.sum())
