"""The one-block select against the multi-launch select, over its thread
counts' edges and every kind of score."""

import numpy as np
import pytest
import torch

import oracle as O
from cacheblend_vllm import _native
from cacheblend_vllm import selection as S

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)


def _scores(kind: str, n: int, rng) -> np.ndarray:
    s = np.exp(rng.normal(size=n)).astype(np.float32)
    if kind == "ties":
        s = rng.integers(0, 5, n).astype(np.float32) - 2.0
    elif kind == "one value":
        s[:] = 0.25
    elif kind == "special":
        for v in (np.nan, np.inf, -np.inf, 0.0, -0.0, np.float32(1e-40), np.finfo(np.float32).min):
            s[rng.random(n) < 0.1] = v
    return s


@pytest.mark.parametrize("n", [1, 8, 9, 2047, 2048, 2049, 8191, 8192, 8193, 16383, 16384, 16385])
@pytest.mark.parametrize("kind", ["spread", "ties", "one value", "special"])
def test_one_block_equals_the_multi_launch_select(n, kind):
    rng = np.random.default_rng(n)
    scores = torch.from_numpy(_scores(kind, n, rng)).to(DEV)
    wide = torch.empty(n + 1, device=DEV)
    wide[1:] = scores
    for gaps in (0.0, 0.1, 1.0):
        gap = torch.from_numpy(rng.random(n) < gaps).to(DEV)
        forced = torch.from_numpy(rng.random(n) < 0.05).to(DEV)
        for f in (None, forced):
            for radius in (0, 1, 16, 4096):
                for ratio in (0.0, 0.15, 1.0):
                    print(f"n={n} {kind} gaps={gaps} forced={f is not None} radius={radius} ratio={ratio}", flush=True)
                    got = S.select(scores, gap, ratio, f, radius)
                    want = S.select(scores, gap, ratio, f, radius, flags=_native.SELECT_MULTI_LAUNCH)
                    assert torch.equal(got, want)
        if kind != "special":
            gap_np = gap.cpu().numpy()
            want = O.select(scores.cpu().numpy(), gap_np, 0.15, O.dilate(gap_np, 16))
            got = S.select(wide[1:], gap, 0.15, None, 16)  # scores 4 bytes off a 16-byte boundary
            np.testing.assert_array_equal(got.cpu().numpy(), want)
