"""The loader's streams in order: its tables go up on the Load stream, and a
commit on any other stream reads the slots only once they are there; the Load
stream reads pages and the RoPE cache only once the serving stream's work
queued before the loader has written them."""

from types import SimpleNamespace

import pytest
import torch

from cacheblend_vllm import synthetic
from cacheblend_vllm.config import CacheBlendConfig
from cacheblend_vllm.host_store import PinnedChunkSlab, PinnedChunkStore
from cacheblend_vllm.loader import PagedBlendLoader
from cacheblend_vllm.types import BlendPlan, BlendSegment

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)


@pytest.mark.parametrize("slots_on", ["cpu", "cuda"])
@pytest.mark.parametrize("streams", [1, 3])
@pytest.mark.parametrize("column", [False, True])  # a column of slots, or a flat list
def test_commits_wait_for_the_slots(slots_on, streams, column):
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
    loader = PagedBlendLoader(layers, PinnedChunkStore(256, 1 << 20), "r", BlendPlan(prefix, end, 0, ()),
                              slots[:, None] if column else slots, block, CacheBlendConfig.from_extra_config({}), load_stream=load)
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


@pytest.mark.parametrize("slots_on", ["cpu", "cuda"])
@pytest.mark.parametrize("zero_copy", [False, True])
def test_loads_see_what_the_serving_stream_had_queued(slots_on, zero_copy):
    heads, dim, block, blocks, chunk, prefix, end, layers = 2, 64, 16, 24, 64, 96, 240, 3
    g = torch.Generator().manual_seed(9)
    pages = [torch.randn(2, blocks, block, heads, dim, generator=g).to(torch.bfloat16).to(DEV) for _ in range(layers)]
    slots = synthetic.block_slots(torch.randperm(blocks, generator=g), block, end).to(slots_on)
    angle = torch.rand(512, dim // 2, generator=g)
    cos_sin = torch.cat([angle.cos(), angle.sin()], dim=-1).to(DEV)
    slab = PinnedChunkSlab((2, chunk, heads, dim), torch.bfloat16, chunks_per_arena=8)
    store = PinnedChunkStore(chunk, 1 << 30, on_release=slab.free)
    sid = store.begin_put("model", 0, list(range(chunk)), layers)
    for layer in range(layers):
        host = slab.alloc()
        host.copy_(torch.randn(2, chunk, heads, dim, generator=g))
        store.put_layer_host(sid, layer, host)
    segments = (BlendSegment(sid, prefix + 32),)
    store.pin("r", segments)
    plan = BlendPlan(prefix, end, chunk, segments)
    config = CacheBlendConfig.from_extra_config({})
    load = torch.cuda.Stream()

    def buffers(kv, cache):
        rope = SimpleNamespace(head_size=dim, rotary_dim=dim, is_neox_style=True, cos_sin_cache=cache)
        loader = PagedBlendLoader(kv, store, "r", plan, slots, block, config, load_stream=load, zero_copy=zero_copy)
        out = []
        loader.prefetch(0, rope)
        for layer in range(layers):
            got = loader.get(layer)
            loader.prefetch(layer + 1, rope)
            out.append(got.clone())
            loader.commit(layer, got)
        return out

    want = buffers([p.clone() for p in pages], cos_sin.clone())
    stale, no_table = [torch.zeros_like(p) for p in pages], torch.zeros_like(cos_sin)
    torch.cuda.synchronize()
    torch.cuda._sleep(20_000_000)
    for old, new in zip(stale, pages):
        old.copy_(new)
    no_table.copy_(cos_sin)
    got = buffers(stale, no_table)
    for a, b in zip(got, want):
        assert torch.equal(a, b)
    store.release("r", None)
    torch.cuda.synchronize()
