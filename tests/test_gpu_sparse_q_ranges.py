"""GPU parity of the Sparse-Q passes at the ends of their row tiles, key
blocks and ranges, against float64."""

import numpy as np
import pytest
import torch

from cacheblend_vllm import _native
from cacheblend_vllm import selection as S

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)


def _f64(q, k, rows, pos, scale):
    """(attention mass per key, largest sum_i |q_i k_i|) in float64."""
    g = q.shape[1] // k.shape[1]
    full, size = np.zeros(k.shape[0]), 0.0
    visible = pos[rows].numpy()[:, None] >= np.arange(k.shape[0])[None, :]
    for h in range(q.shape[1]):
        qh, kh = q[rows, h].double().numpy(), k[:, h // g].double().numpy()
        x = np.where(visible, qh @ kh.T * scale, -np.inf)
        e = np.exp(x - x.max(axis=1, keepdims=True, initial=-1e300))
        full += (e / np.maximum(e.sum(axis=1, keepdims=True), 1e-300)).sum(axis=0)
        size = max(size, float((np.abs(qh) @ np.abs(kh).T).max()))
    return full, size


# query rows around the 64-row tile and the 32-row block, keys around the
# 32-key block and 64-key tile, head sizes around the padded 64 and 128 (and
# one above), rows in any order and at positions before the first key
@pytest.mark.parametrize("nq,nk,hq,hkv,d", [
    (1, 1, 1, 1, 64), (1, 65, 16, 1, 128), (31, 64, 2, 1, 64), (33, 63, 2, 2, 128), (65, 700, 3, 1, 100),
    (22, 1031, 6, 2, 3), (64, 4097, 8, 4, 128), (130, 2047, 16, 8, 128), (40, 333, 10, 2, 66), (9, 200, 4, 2, 136),
])
def test_f32_matches_float64(nq, nk, hq, hkv, d):
    g = torch.Generator().manual_seed(nq + nk)
    n = 2 * nq
    q, k = torch.randn(n, hq, d, generator=g), torch.randn(nk, hkv, d, generator=g)
    pos = torch.randint(-1, nk, (n,), generator=g)
    rows = torch.randperm(n, generator=g)[:nq]
    pos[rows[0]] = nk - 1
    scale = d ** -0.5
    _, full = S.sparse_q_full_scores(q.to(DEV), k.to(DEV), rows.to(DEV), pos.to(DEV), scale, want_full=True)
    want, size = _f64(q, k, rows, pos, scale)
    # every term is positive; a logit is off by at most (d + 3) roundings of
    # its absolute terms, twice in a probability (itself and its row's sum),
    # and the row's sum, the exponentials and the score's sum by the rest
    u = 2.0 ** -24
    bound = np.expm1(2 * (d + 3) * u * size * scale) + (nk + nq * hq + 24 + 2 * size * scale) * u
    err = np.abs(full.cpu().numpy() - want) / np.maximum(want, 1e-300)
    print(f"largest error / bound {err.max() / bound:.3f}", flush=True)
    assert err.max() <= bound


def test_f32_unaligned_views():
    # rows 4 bytes off a 16-byte boundary
    nq, nk, hq, hkv, d = 50, 500, 4, 2, 64
    g = torch.Generator().manual_seed(4)
    q, k = torch.randn(nq, hq, d, generator=g), torch.randn(nk, hkv, d, generator=g)
    pos = torch.arange(nk - nq, nk)

    def off(t):
        flat = torch.zeros(t.shape[0], t.shape[1] * d + 1)
        flat[:, 1:] = t.reshape(t.shape[0], -1)
        return flat.to(DEV)[:, 1:].unflatten(1, (t.shape[1], d))

    _, want = S.sparse_q_full_scores(q.to(DEV), k.to(DEV), None, pos.to(DEV), 0.125, want_full=True)
    _, got = S.sparse_q_full_scores(off(q), off(k), None, pos.to(DEV), 0.125, want_full=True)
    assert torch.equal(got, want)


def test_f32_more_keys_than_the_column_pass_holds():
    # 2^31 (key, KV head) pairs: only the first keys are seen, and read
    nk, hkv, seen, lib = (1 << 30) - 1, 2, 100, _native.load()
    g = torch.Generator().manual_seed(1)
    k = torch.empty(nk, hkv, 1, device=DEV)
    first = torch.randn(seen + 1, hkv, 1, generator=g)
    k[:seen + 1] = first.to(DEV)
    q, pos = torch.randn(1, hkv, 1, generator=g), torch.tensor([seen])
    index = torch.tensor([*range(seen + 2), 1 << 29, nk - 1], device=DEV)
    out = torch.empty(index.numel(), device=DEV)
    ws = torch.empty(lib.cbk_sparse_q_workspace_bytes(1, nk, hkv, hkv), dtype=torch.uint8, device=DEV)
    dq, dp = q.to(DEV), pos.to(DEV)
    rc = lib.cbk_sparse_q_scores(
        dq.data_ptr(), hkv, None, 1, dp.data_ptr(), k.data_ptr(), hkv, nk, hkv, hkv, 1, 1.0,
        _native.DTYPE_CODES[torch.float32], 0, index.data_ptr(), index.numel(), out.data_ptr(), None,
        ws.data_ptr(), ws.numel(), _native.stream_handle(DEV))
    _native.check(rc, "sparse_q_scores")
    want, _ = _f64(q, first, torch.tensor([0]), pos, 1.0)
    got = out.cpu().numpy()
    del k, ws
    torch.cuda.empty_cache()
    # one product, ~100 exponentials and their sum, each within a few 2^-24
    assert np.all(np.abs(got[:seen + 1] - want) <= 300 * 2.0 ** -24 * want)
    assert np.all(got[seen + 1:] == 0)


# few rows over many keys: up to 64 key ranges (more than the merge's batch of
# loads per wave, ranges without a block, and key counts around a block), column
# units in one to four ranges; entries in {-1, 0, 1} / 8, whose dot products
# are exact in the input type
@pytest.mark.parametrize("nq,nk,hq,hkv,d,dtype", [
    (1, 16385, 1, 1, 64, torch.bfloat16), (64, 9001, 4, 1, 128, torch.bfloat16), (17, 4095, 8, 1, 64, torch.float16),
    (64, 700, 3, 1, 128, torch.float16), (200, 2050, 2, 2, 128, torch.bfloat16), (33, 6000, 16, 1, 64, torch.bfloat16),
])
def test_16_bit_matches_float64(nq, nk, hq, hkv, d, dtype):
    g = torch.Generator().manual_seed(nq + nk)
    q, k = ((torch.randint(-1, 2, (n, h, d), generator=g) / 8).to(dtype) for n, h in ((nq, hq), (nk, hkv)))
    pos = torch.randint(0, nk, (nq,), generator=g).sort().values
    pos[-1] = nk - 1
    rows = torch.arange(nq)
    _, full = S.sparse_q_full_scores(q.to(DEV), k.to(DEV), None, pos.to(DEV), 1.0, want_full=True)
    want, size = _f64(q, k, rows, pos, 1.0)
    # exact logits: the float32 exponentials and sums of positive terms only
    bound = (nk + nq * hq + 24 + 4 * size) * 2.0 ** -24
    err = np.abs(full.cpu().numpy() - want) / np.maximum(want, 1e-300)
    print(f"largest error / bound {err.max() / bound:.3f}", flush=True)
    assert err.max() <= bound
