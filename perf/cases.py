"""The work whose speed matters to a user of this package, as timed cases.

A request that reuses cached KV goes through these calls, in this order: the
store gathers the prompt's KV rows from the pages, a later request loads the
stored chunks and blends them into its pages, the check layer selects the
tokens to recompute (K deviation or Sparse-Q), and every later layer attends
from those tokens only. Shapes are those of the Qwen3 layers that bench.py
and the tests use (0.6B / 1.7B: 16 query heads over 8 KV heads; 8B: 32 over
8; 14B: 40 over 8; 30B-A3B: 32 over 4; head size 128) and, in the drawn
cases, a head size of 64.

``listed()`` names twelve cases, ``draw(rng)`` makes more of the same ranges.
"""

from __future__ import annotations

import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.getcwd(), "pic-kvcache_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from cacheblend_vllm import kv_layout, synthetic  # noqa: E402
from cacheblend_vllm.attention import blend_attention  # noqa: E402
from cacheblend_vllm.config import CacheBlendConfig  # noqa: E402
from cacheblend_vllm.host_store import PinnedChunkSlab, PinnedChunkStore  # noqa: E402
from cacheblend_vllm.loader import PagedBlendLoader  # noqa: E402
from cacheblend_vllm.selection import BlendSelector, kdev_select  # noqa: E402
from cacheblend_vllm.types import BlendPlan, BlendSegment  # noqa: E402

DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
BYTES = {"bf16": 2, "f16": 2, "f32": 4}
BLOCK = 16   # tokens per vLLM block
CHUNK = 256  # tokens per stored chunk


def listed() -> list[dict]:
    return [
        # one layer's rows of a short prompt out of the pages: what the store
        # does after each layer of a prefill, at its smallest
        dict(name="gather_layer_333", kind="gather", dtype="bf16", layers=1, tokens=333, heads=8, dim=128,
             layout="merged_first"),
        # all 36 layers of an 8K prompt back into the pages: a stored prompt
        # loaded whole
        dict(name="scatter_36_layers_8k", kind="scatter", dtype="bf16", layers=36, tokens=8192, heads=8, dim=128,
             layout="merged_first"),
        # a request's layerwise load: stored chunks over the host link, K
        # moved to new positions, blended with the cached prefix, committed
        dict(name="blend_load_8_layers", kind="blend_load", dtype="bf16", layers=8, tokens=7167, prefix=512,
             heads=4, dim=128, neox=True),
        # K-deviation selection of a short prompt on one of two ranks (4 KV
        # heads split over them), and of a long one
        dict(name="kdev_1537", kind="kdev", dtype="f16", tokens=1537, prefix=256, heads=2, dim=128, radius=0,
             ratio=0.15),
        dict(name="kdev_65536", kind="kdev", dtype="bf16", tokens=65536, prefix=0, heads=4, dim=128, radius=16,
             ratio=0.15),
        # Sparse-Q scores: a fully cached 16K prompt, where the last 64
        # tokens are the queries (the configuration's default), and a 96K
        # prompt with 4096 tokens that no chunk covers
        dict(name="sparse_q_tail_16k", kind="sparse_q", dtype="bf16", keys=16383, queries=0, q_heads=32, heads=8,
             dim=128),
        dict(name="sparse_q_96k", kind="sparse_q", dtype="bf16", keys=98304, queries=4096, q_heads=32, heads=4,
             dim=128),
        # attention of the selected tokens: few tokens of a well-covered 8K
        # prompt, an ordinary 4K prompt (its gaps and 15% of the rest), and
        # the long prompt of the blend load benchmark
        dict(name="attention_180_of_8k", kind="attention", dtype="bf16", queries=180, keys=8191, q_heads=32,
             heads=8, dim=128),
        dict(name="attention_990_of_4k", kind="attention", dtype="f16", queries=990, keys=4095, q_heads=32,
             heads=8, dim=128),
        dict(name="attention_7000_of_32k", kind="attention", dtype="bf16", queries=7000, keys=32767, q_heads=32,
             heads=4, dim=128),
        # float32 models, as the accuracy comparisons run them: the same two
        # steps on a 2K prompt of a 16-over-8-head layer
        dict(name="attention_f32_500_of_2k", kind="attention", dtype="f32", queries=500, keys=2047, q_heads=16,
             heads=8, dim=128),
        dict(name="sparse_q_f32_2k", kind="sparse_q", dtype="f32", keys=2047, queries=256, q_heads=16, heads=8,
             dim=128),
    ]


# the most (queries x keys x query heads) of a drawn case, and of a float32
# Sparse-Q one the most queries of one KV head, so that none costs more than
# the largest listed one
_MOST_LOGITS = {"bf16": 4096 * 98304 * 32 // 2, "f16": 4096 * 98304 * 32 // 2, "f32": 500 * 2047 * 16}
_MOST_F32_ROWS = 400


def _log_int(rng, lo: int, hi: int) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng) -> dict:
    kind = rng.choice(["gather", "scatter", "blend_load", "kdev", "kdev", "sparse_q", "sparse_q", "sparse_q",
                       "attention", "attention", "attention"])
    dim = rng.choice([128, 128, 64])
    heads = rng.choice([2, 4, 8])
    dtype = rng.choice(["bf16", "bf16", "f16", "f32"])
    if kind in ("gather", "scatter"):
        layers = rng.choice([1, 1, 28, 36])
        return dict(kind=kind, dtype=dtype, layers=layers, tokens=_log_int(rng, 16, 32768 if layers == 1 else 4096),
                    heads=heads, dim=dim, layout=rng.choice(["merged_first", "merged_block", "separate"]))
    if kind == "blend_load":
        tokens = _log_int(rng, 1500, 7167)
        return dict(kind=kind, dtype=rng.choice(["bf16", "f16"]), layers=rng.choice([4, 8]), tokens=tokens,
                    prefix=BLOCK * rng.randrange(0, 33), heads=rng.choice([2, 4]), dim=dim,
                    neox=rng.choice([True, True, False]))
    if kind == "kdev":
        return dict(kind=kind, dtype=dtype, tokens=_log_int(rng, 300, 65536), prefix=BLOCK * rng.randrange(0, 65),
                    heads=heads if dtype != "f32" else min(heads, 4), dim=dim, radius=rng.choice([0, 16]),
                    ratio=rng.choice([0.05, 0.15, 0.3]))
    q_heads, heads = rng.choice([(16, 8), (32, 8), (40, 8), (32, 4), (8, 2)])
    f32 = dtype == "f32"
    keys = _log_int(rng, 700, 2047 if f32 else 98304 if kind == "sparse_q" else 32767)
    most = min(keys // 3, 500 if f32 else 4096, _MOST_LOGITS[dtype] // (keys * q_heads))
    if f32 and kind == "sparse_q":
        most = min(most, _MOST_F32_ROWS * heads // q_heads)
    queries = _log_int(rng, 20, most)
    if kind == "sparse_q" and rng.random() < 0.4:
        queries = 0  # fully cached
    return dict(kind=kind, dtype=dtype, keys=keys, queries=queries, q_heads=q_heads, heads=heads, dim=dim)


# ------------------------------------------------------------------ inputs


class _Rope:
    """What the loader reads of a model's rotary embedding."""

    def __init__(self, dim: int, positions: int, neox: bool):
        self.head_size = self.rotary_dim = dim
        self.is_neox_style = neox
        inv = 1.0 / (1e6 ** (torch.arange(0, dim, 2, dtype=torch.float32) / dim))
        angle = torch.arange(positions, dtype=torch.float32)[:, None] * inv
        self.cos_sin_cache = torch.cat([angle.cos(), angle.sin()], dim=-1).cuda()


def _randn(g: torch.Generator, *shape: int, dtype: torch.dtype) -> torch.Tensor:
    return torch.randn(shape, generator=g, device="cuda", dtype=dtype)


def _pages(g, layout: str, blocks: int, heads: int, dim: int, dtype):
    if layout == "merged_block":
        return _randn(g, blocks, 2, BLOCK, heads, dim, dtype=dtype)
    pool = _randn(g, 2, blocks, BLOCK, heads, dim, dtype=dtype)
    return pool if layout == "merged_first" else (pool[0], pool[1])


def _slots(seed: int, blocks: int, tokens: int) -> torch.Tensor:
    order = torch.from_numpy(np.random.default_rng(seed).permutation(blocks))
    return synthetic.block_slots(order, BLOCK, tokens)


def _segments(case: dict, seed: int) -> list[tuple[int, int, int]]:
    """(source start, target start, tokens) of the stored segments a prompt
    reuses after its prefix: whole chunks, one to six of them together, apart
    by gaps of 1 to 300 tokens."""
    rng = np.random.default_rng(seed)
    found, at, source = [], case["prefix"], 0
    while True:
        at += int(rng.integers(1, 301))
        n = CHUNK * min(int(rng.integers(1, 7)), (case["tokens"] - 1 - at) // CHUNK)
        if n <= 0:
            return found
        found.append((source, at, n))
        at += n
        source += n + 512


def _blend_load(case: dict, seed: int, g) -> dict:
    dtype, heads, dim, end = DTYPES[case["dtype"]], case["heads"], case["dim"], case["tokens"]
    # the gaps between segments belong to the request: the plan is drawn from
    # the sizes, so that every seed's inputs have the same shapes
    segments = _segments(case, 17)
    hits = sum(n for _, _, n in segments)
    blocks = (end + BLOCK - 1) // BLOCK + 8
    layers = [_pages(g, "merged_first", blocks, heads, dim, dtype) for _ in range(case["layers"])]
    slab = PinnedChunkSlab((2, CHUNK, heads, dim), dtype, chunks_per_arena=max(64, hits // CHUNK))
    store = PinnedChunkStore(CHUNK, 1 << 40, on_release=slab.free)
    runs = [slab.alloc_run(hits // CHUNK) for _ in layers]
    for run in runs:
        for chunk in run:
            chunk.copy_(_randn(g, 2, CHUNK, heads, dim, dtype=dtype))
    pieces, k = [], 0
    for i, (source, target, n) in enumerate(segments):
        for c in range(0, n, CHUNK):
            first = source + c + 7 * i
            sid = store.begin_put("model", source + c, list(range(first, first + CHUNK)), len(layers))
            for layer, run in enumerate(runs):
                store.put_layer_host(sid, layer, run[k])
            pieces.append(BlendSegment(sid, target + c))
            k += 1
    store.pin("request", pieces)
    return dict(layers=layers, slab=slab, store=store, runs=runs, segments=segments,
                plan=BlendPlan(case["prefix"], end, hits, tuple(pieces)), slots=_slots(seed, blocks, end),
                rope=_Rope(dim, 16384, case["neox"]), config=CacheBlendConfig.from_extra_config({}))


def prepare(case: dict, seed: int) -> dict:
    g = torch.Generator(device="cuda").manual_seed(seed)
    kind, dtype, heads, dim = case["kind"], DTYPES[case["dtype"]], case["heads"], case["dim"]
    if kind in ("gather", "scatter"):
        # as many pages again as the prompt fills, in random order
        blocks = 2 * ((case["tokens"] + BLOCK - 1) // BLOCK) + 8
        pages = [_pages(g, case["layout"], blocks, heads, dim, dtype) for _ in range(case["layers"])]
        state = dict(kind=kind, pages=pages, slots=_slots(seed, blocks, case["tokens"]).cuda())
        if case["layers"] > 1:
            state["cache"] = kv_layout.PagedKVCache(pages, BLOCK)
        if kind == "scatter":
            lead = (case["layers"],) if case["layers"] > 1 else ()
            state["rows"] = _randn(g, *lead, 2, case["tokens"], heads, dim, dtype=dtype)
        return state
    if kind == "blend_load":
        return dict(kind=kind, **_blend_load(case, seed, g))
    if kind == "kdev":
        n, width = case["tokens"], heads * dim
        # one gap layout per size, so that every seed selects as many tokens
        gap = torch.from_numpy(synthetic.gap_layout(n, 5)).cuda()
        cached = _randn(g, case["prefix"] + n, width, dtype=torch.float32)
        old = cached[case["prefix"]:]
        old[gap] = 0
        # chunks computed in another context: most keys barely moved, few a lot
        sigma = 0.02 * torch.exp(_randn(g, n, 1, dtype=torch.float32))
        fresh = old + sigma * _randn(g, n, width, dtype=torch.float32)
        fresh[gap] = _randn(g, int(gap.sum()), width, dtype=torch.float32)
        index = torch.arange(case["prefix"], case["prefix"] + n, device="cuda")
        return dict(kind=kind, fresh=fresh.to(dtype), cached=cached.to(dtype), index=index, gap=gap,
                    ratio=case["ratio"], radius=case["radius"])
    # queries and keys as a layer's RMS norms leave them: N(0, 1) entries
    q_heads, keys = case["q_heads"], case["keys"]
    key = _randn(g, keys, heads, dim, dtype=dtype)
    if kind == "sparse_q":
        gap = np.zeros(keys, dtype=bool)
        if case["queries"]:
            gap = synthetic.sparse_q_layout(keys, case["queries"], seed)
        config = CacheBlendConfig.from_extra_config({"selection_strategy": "sparse_q"})
        return dict(kind=kind, selector=BlendSelector(config, BLOCK), key=key, scale=dim ** -0.5,
                    query=_randn(g, keys, q_heads, dim, dtype=dtype), index=torch.arange(keys, device="cuda"),
                    gap=torch.from_numpy(gap).cuda())
    rng = np.random.default_rng(seed)
    # the selected tokens lie past a cached prefix of a sixteenth, the last
    # token always among them
    chosen = rng.choice(np.arange(keys // 16, keys - 1), case["queries"] - 1, replace=False)
    positions = torch.from_numpy(np.sort(np.append(chosen, keys - 1))).cuda()
    return dict(kind=kind, query=_randn(g, case["queries"], q_heads, dim, dtype=dtype), key=key,
                value=_randn(g, keys, heads, dim, dtype=dtype), positions=positions, scale=dim ** -0.5)


# -------------------------------------------------------------------- pass


def run(state: dict):
    kind = state["kind"]
    if kind == "gather":
        if "cache" in state:
            return state["cache"].gather(state["slots"])
        return kv_layout.gather_paged_kv(state["pages"][0], state["slots"], BLOCK)
    if kind == "scatter":
        if "cache" in state:
            state["cache"].scatter(state["rows"], state["slots"])
        else:
            kv_layout.scatter_paged_kv(state["rows"], state["pages"][0], state["slots"], BLOCK)
        return [list(p) if isinstance(p, tuple) else p for p in state["pages"]]
    if kind == "blend_load":
        layers = state["layers"]
        loader = PagedBlendLoader(layers, state["store"], "request", state["plan"], state["slots"], BLOCK,
                                  state["config"])
        loader.prefetch(0, state["rope"])
        for layer in range(len(layers)):
            buffer = loader.get(layer)
            loader.prefetch(layer + 1, state["rope"])
            loader.commit(layer, buffer)
        return list(layers)
    if kind == "kdev":
        selected, scores = kdev_select(state["fresh"], state["cached"], state["index"], state["gap"],
                                       state["ratio"], state["radius"])
        return {"selected": selected, "scores": scores}
    if kind == "sparse_q":
        scores, forced, _ = state["selector"]._sparse_q_scores(state["query"], state["key"], state["index"],
                                                               state["gap"], state["scale"])
        return {"scores": scores, "forced": forced}
    return blend_attention(state["query"], state["key"], state["value"], state["positions"], state["scale"])


# ----------------------------------------------------- work and exact values


def _visible(case: dict, seed: int = 0) -> float:
    """(query, key) pairs a causal pass looks at."""
    keys = case["keys"]
    if case["kind"] == "attention":  # positions uniform over (keys / 16, keys)
        return case["queries"] * (keys / 16 + keys) / 2
    if case["queries"]:
        return float((np.flatnonzero(synthetic.sparse_q_layout(keys, case["queries"], seed)) + 1).sum())
    tail = min(64, keys)
    return tail * (keys - (tail - 1) / 2)


def work(case: dict) -> dict:
    kind, es = case["kind"], BYTES[case["dtype"]]
    row = case["heads"] * case["dim"] * es
    if kind in ("gather", "scatter"):
        return {"bytes": 2 * case["layers"] * 2 * case["tokens"] * row + 8 * case["tokens"], "flops": 0}
    if kind == "blend_load":
        # every committed row written once, the hit rows read once
        hits = sum(n for _, _, n in _segments(case, 17))
        return {"bytes": case["layers"] * 2 * (hits + case["tokens"] - case["prefix"]) * row, "flops": 0}
    if kind == "kdev":
        n = case["tokens"]
        return {"bytes": 2 * n * row + 13 * n, "flops": 3 * n * case["heads"] * case["dim"]}
    queries = case["queries"] or min(64, case["keys"])
    q_row = case["q_heads"] * case["dim"] * es
    products = 2.0 * case["dim"] * case["q_heads"] * _visible(case)
    if kind == "sparse_q":
        return {"bytes": queries * q_row + case["keys"] * (row + 4), "flops": products}
    return {"bytes": 2 * queries * q_row + 2 * case["keys"] * row, "flops": 2 * products}


def tolerance(case: dict):
    kind, dtype = case["kind"], case["dtype"]
    if kind in ("gather", "scatter", "blend_load"):
        return "exact"
    if kind == "kdev":
        return {"rel": 1e-6, "max": 1e-5}
    if kind == "sparse_q":
        # the logits are rounded to the input type, as the reference's matmul
        # output is; the scores sum many of them in float32
        return {"rel": {"bf16": 1e-3, "f16": 1.5e-4, "f32": 1e-5}[dtype]}
    return {"rel": {"bf16": 1e-2, "f16": 3e-3, "f32": 1e-5}[dtype]}


def _exact_scores(state: dict, case: dict):
    keys, group = case["keys"], case["q_heads"] // case["heads"]
    rows = torch.nonzero(state["gap"]).flatten()
    if not rows.numel():
        rows = torch.arange(max(0, keys - 64), keys, device="cuda")
    full = torch.zeros(keys, dtype=torch.float64, device="cuda")
    place = torch.arange(keys, device="cuda")
    step = max(1, (1 << 27) // keys)
    for h in range(case["q_heads"]):
        k = state["key"][:, h // group].double().t().contiguous()
        for part in rows.split(step):
            logits = (state["query"][part, h].double() @ k) * state["scale"]
            logits.masked_fill_(place[None, :] > part[:, None], -math.inf)
            full += torch.softmax(logits, dim=1).sum(dim=0)
    return {"scores": full, "forced": None}


def _exact_attention(state: dict, case: dict) -> torch.Tensor:
    keys, group = case["keys"], case["q_heads"] // case["heads"]
    out = torch.empty(state["query"].shape, dtype=torch.float64, device="cuda")
    place = torch.arange(keys, device="cuda")
    step = max(1, (1 << 27) // keys)
    for h in range(case["q_heads"]):
        k = state["key"][:, h // group].double().t().contiguous()
        v = state["value"][:, h // group].double().contiguous()
        for lo in range(0, case["queries"], step):
            positions = state["positions"][lo:lo + step]
            logits = (state["query"][lo:lo + step, h].double() @ k) * state["scale"]
            logits.masked_fill_(place[None, :] > positions[:, None], -math.inf)
            out[lo:lo + step, h] = torch.softmax(logits, dim=1) @ v
    return out


def _exact_load(state: dict, case: dict) -> list:
    dim, neox = case["dim"], case["neox"]
    cos, sin = state["rope"].cos_sin_cache.double().chunk(2, dim=-1)
    slots = state["slots"].cuda()
    result = []
    for layer, run in zip(state["layers"], state["runs"]):
        pages = layer.double().reshape(2, -1, *layer.shape[3:])
        pages[:, slots[case["prefix"]:]] = 0
        rows = torch.cat([chunk.cuda() for chunk in run], dim=1).double()
        at = 0
        for source, target, n in state["segments"]:
            old = torch.arange(source, source + n, device="cuda")
            new = torch.arange(target, target + n, device="cuda")
            c = (cos[new] * cos[old] + sin[new] * sin[old])[:, None]
            s = (sin[new] * cos[old] - cos[new] * sin[old])[:, None]
            k = rows[0, at:at + n]
            a, b = (k[..., :dim // 2], k[..., dim // 2:]) if neox else (k[..., 0::2], k[..., 1::2])
            a, b = a * c - b * s, b * c + a * s
            k = torch.cat([a, b], dim=-1) if neox else torch.stack([a, b], dim=-1).flatten(-2)
            pages[0, slots[new]] = k
            pages[1, slots[new]] = rows[1, at:at + n]
            at += n
        result.append(pages.reshape(layer.shape))
    return result


def exact(case: dict, seed: int):
    kind = case["kind"]
    if kind in ("gather", "scatter"):
        return None  # copies
    state = prepare(case, seed)
    if kind == "blend_load":
        return _exact_load(state, case)
    if kind == "kdev":
        old = state["cached"][state["index"]].double()
        return {"selected": None, "scores": (state["fresh"].double() - old).square().sum(dim=1)}
    if kind == "sparse_q":
        return _exact_scores(state, case)
    return _exact_attention(state, case)
