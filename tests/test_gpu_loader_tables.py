"""The loader's tables go up on the Load stream: a commit on any other stream
reads the slots only once they are there."""

import pytest
import torch

from cacheblend_vllm import synthetic
from cacheblend_vllm.config import CacheBlendConfig
from cacheblend_vllm.host_store import PinnedChunkStore
from cacheblend_vllm.loader import PagedBlendLoader
from cacheblend_vllm.types import BlendPlan

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)


@pytest.mark.parametrize("slots_on", ["cpu", "cuda"])
@pytest.mark.parametrize("streams", [1, 3])
def test_commits_wait_for_the_slots(slots_on, streams):
    heads, dim, block, blocks, end, prefix = 2, 64, 16, 40, 333, 32
    g = torch.Generator().manual_seed(7)
    load = torch.cuda.Stream()
    serving = [torch.cuda.Stream() for _ in range(streams)]
    layers = [torch.zeros(2, blocks, block, heads, dim, dtype=torch.bfloat16, device=DEV) for _ in serving]
    rows = [torch.randn(2, end, heads, dim, generator=g).to(torch.bfloat16).to(DEV) for _ in serving]
    slots = synthetic.block_slots(torch.randperm(blocks, generator=g), block, end).to(slots_on)
    # memory that a missing wait would read instead of the slots
    junk = [torch.full((4096,), -1, dtype=torch.int32, device=DEV) for _ in range(8)]
    torch.cuda.synchronize()
    del junk
    with torch.cuda.stream(load):
        torch.cuda._sleep(20_000_000)
    loader = PagedBlendLoader(layers, PinnedChunkStore(256, 1 << 20), "r", BlendPlan(prefix, end, 0, ()), slots,
                              block, CacheBlendConfig.from_extra_config({}), load_stream=load)
    for i, stream in enumerate(serving):
        with torch.cuda.stream(stream):
            loader.commit(i, rows[i])
    del loader  # its tables are freed while the copies may still be queued
    fill = torch.full((4096,), -1, dtype=torch.int32, device=DEV)
    torch.cuda.synchronize()
    assert int(fill.sum()) == -4096
    for layer, want in zip(layers, rows):
        flat = layer.reshape(2, -1, heads, dim)
        assert torch.equal(flat[:, slots[prefix:].to(DEV)], want[:, prefix:])
        assert int(torch.count_nonzero(flat.float().abs().sum((0, 2, 3)))) == end - prefix
