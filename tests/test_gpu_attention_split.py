"""GPU parity of the attention kernels' row tiles, key blocks and key ranges,
at the sizes where they end unevenly, against float64."""

import numpy as np
import pytest
import torch

from cacheblend_vllm import _native
from cacheblend_vllm.attention import blend_attention

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)


def _f64(q, k, v, pos, scale):
    """(outputs, sum_k p_k |v_k|, largest sum_i |q_i k_i|) in float64."""
    nq, hq, d = q.shape
    g = hq // k.shape[1]
    out, mass, size = np.zeros((nq, hq, d)), np.zeros((nq, hq, d)), 0.0
    visible = pos.numpy()[:, None] >= np.arange(k.shape[0])[None, :]
    for h in range(hq):
        qh, kh, vh = (t.double().numpy() for t in (q[:, h], k[:, h // g], v[:, h // g]))
        x = np.where(visible, qh @ kh.T * scale, -np.inf)
        e = np.exp(x - x.max(axis=1, keepdims=True, initial=-1e300))
        p = e / np.maximum(e.sum(axis=1, keepdims=True), 1e-300)
        out[:, h], mass[:, h] = p @ vh, p @ np.abs(vh)
        size = max(size, float((np.abs(qh) @ np.abs(kh).T).max()))
    return out, mass, size


def _f32_bound(mass, size, d, nk, scale):
    """What float32 can move an output by: a logit by (d + 3) roundings of at
    most 2^-24 of its absolute terms, hence its probability by that factor (and
    the sum it is divided by, once more), and each of the two sums over nk keys
    and the exponential by at most (nk + 8) roundings."""
    u = 2.0 ** -24
    return (2 * np.expm1((d + 3) * u * size * scale) + 2 * (nk + 8) * u) * mass + 1e-30


def _inputs(nq, nk, hq, hkv, d, dtype=torch.float32, seed=0):
    g = torch.Generator().manual_seed(seed)
    q, k, v = (torch.randn(n, h, d, generator=g).to(dtype) for n, h in ((nq, hq), (nk, hkv), (nk, hkv)))
    pos = torch.randint(0, nk, (nq,), generator=g)
    pos[-1] = nk - 1
    return q, k, v, pos


# rows of (query, group head) around the 64-row tile, keys around the 32-key
# block, head sizes around the padded 64 and 128, and more ranges than a tile
# with few keys has blocks
@pytest.mark.parametrize("nq,nk,hq,hkv,d", [
    (1, 1, 1, 1, 128), (1, 33, 2, 1, 64), (16, 32, 4, 1, 128), (63, 300, 2, 2, 64), (65, 257, 3, 1, 128),
    (22, 1031, 6, 2, 100), (5, 4099, 8, 8, 128), (9, 700, 4, 2, 3), (40, 513, 4, 4, 66), (130, 2047, 16, 8, 128),
])
def test_f32_matches_float64(nq, nk, hq, hkv, d):
    q, k, v, pos = _inputs(nq, nk, hq, hkv, d)
    scale = d ** -0.5
    got = blend_attention(q.to(DEV), k.to(DEV), v.to(DEV), pos.to(DEV), scale).cpu().numpy()
    want, mass, size = _f64(q, k, v, pos, scale)
    err = np.abs(got - want)
    print(f"largest error / bound {(err / _f32_bound(mass, size, d, nk, scale)).max():.3f}", flush=True)
    assert np.all(err <= _f32_bound(mass, size, d, nk, scale))


def test_f32_unaligned_views_and_one_range():
    # rows 4 bytes off a 16-byte boundary, and the entry without a workspace
    nq, nk, hq, hkv, d = 37, 901, 4, 2, 64
    q, k, v, pos = _inputs(nq, nk, hq, hkv, d, seed=1)
    want, mass, size = _f64(q, k, v, pos, 0.125)
    bound = _f32_bound(mass, size, d, nk, 0.125)

    def off(t):
        flat = torch.zeros(t.shape[0], t.shape[1] * d + 1)
        flat[:, 1:] = t.reshape(t.shape[0], -1)
        return flat.to(DEV)[:, 1:].unflatten(1, (t.shape[1], d))

    got = blend_attention(off(q), off(k), off(v), pos.to(DEV), 0.125).cpu().numpy()
    assert np.all(np.abs(got - want) <= bound)
    dq, dk, dv, dp = (t.to(DEV) for t in (q, k, v, pos))
    out = torch.empty_like(dq)
    rc = _native.load().cbk_blend_attention(
        dq.data_ptr(), hq * d, dp.data_ptr(), nq, dk.data_ptr(), hkv * d, dv.data_ptr(), hkv * d, nk, hq, hkv, d,
        0.125, _native.DTYPE_CODES[torch.float32], out.data_ptr(), hq * d, _native.stream_handle(DEV))
    _native.check(rc, "blend_attention")
    assert np.all(np.abs(out.cpu().numpy() - want) <= bound)


def test_f32_values_past_a_position_do_not_reach_its_row():
    # keys and values past each position hold NaN and infinities; rows that
    # see one have it in their result; a position below 0 sees nothing
    nq, nk, hq, hkv, d = 20, 400, 2, 1, 64
    q, k, v, _ = _inputs(nq, nk, hq, hkv, d, seed=2)
    pos = torch.arange(nq) * 20 - 1
    want, mass, size = _f64(q, k, v, pos.clamp(min=0), 0.125)
    k[300], v[300], v[310, 0, 5], k[330] = float("nan"), float("inf"), float("nan"), float("inf")
    got = blend_attention(q.to(DEV), k.to(DEV), v.to(DEV), pos.to(DEV), 0.125).cpu().numpy()
    clean = (pos.numpy() < 300) & (pos.numpy() >= 0)
    assert np.all(np.abs(got - want)[clean] <= _f32_bound(mass, size, d, nk, 0.125)[clean])
    assert np.all(got[pos.numpy() < 0] == 0)
    assert np.all(np.isnan(got[pos.numpy() >= 300]))


def _attend_in_guards(q, k, v, pos, scale, ranges):
    """``blend_attention`` through the C entry, ``out`` and the ranges' scratch
    inside larger buffers: (out, whether the memory around both is untouched)."""
    lib, (nq, hq, d), (nk, hkv, _) = _native.load(), q.shape, k.shape
    code, guard = _native.DTYPE_CODES[q.dtype], 1 << 16
    nbytes = lib.cbk_blend_attention_workspace_bytes(nq, nk, hq, hkv, d, code) if ranges else 0
    assert (nbytes > 0) == ranges
    out_bytes = nq * hq * d * q.element_size()
    bufs = [torch.full((2 * guard + n,), 0x5A, dtype=torch.uint8, device=DEV) for n in (out_bytes, nbytes)]
    out = bufs[0][guard:guard + out_bytes].view(q.dtype).view(nq, hq, d)
    rc = lib.cbk_blend_attention_ws(
        q.data_ptr(), hq * d, pos.data_ptr(), nq, k.data_ptr(), hkv * d, v.data_ptr(), hkv * d, nk, hq, hkv, d,
        scale, code, out.data_ptr(), hq * d, bufs[1].data_ptr() + guard if ranges else None, nbytes,
        _native.stream_handle(DEV))
    _native.check(rc, "blend_attention")
    whole = all(bool((b[:guard] == 0x5A).all()) and bool((b[-guard:] == 0x5A).all()) for b in bufs)
    return out.cpu(), whole


# a last row tile with and without rows past the end, the bad key in the
# first, a middle and the last range of the last tile, and past the positions of the first
@pytest.mark.parametrize("ranges", [False, True])
@pytest.mark.parametrize("bad_key", [20, 500, 890])
@pytest.mark.parametrize("nq,d", [(36, 64), (36, 66), (37, 128), (40, 64), (5, 100)])
def test_f32_keys_that_are_not_finite_reach_the_rows_that_see_them_only(nq, d, bad_key, ranges):
    nk, hq, hkv, scale = 900, 4, 2, 0.125
    q, k, v, _ = _inputs(nq, nk, hq, hkv, d, seed=nq)
    pos = torch.linspace(-1, nk - 1, nq).long()
    want, mass, size = _f64(q, k, v, pos.clamp(min=0), scale)
    k[bad_key, 0], v[bad_key, 1] = float("nan"), float("inf")
    print(f"nq={nq} d={d} bad={bad_key} ranges={ranges}", flush=True)
    got, whole = _attend_in_guards(*(t.to(DEV) for t in (q, k, v, pos)), scale, ranges)
    assert whole
    got, sees = got.numpy(), pos.numpy() >= bad_key
    clean = ~sees & (pos.numpy() >= 0)
    assert np.all(np.abs(got - want)[clean] <= _f32_bound(mass, size, d, nk, scale)[clean])
    assert np.all(got[pos.numpy() < 0] == 0)
    assert np.all(np.isnan(got[sees, :2])) and np.all(np.isposinf(got[sees, 2:]))


# logits around the type's lowest and largest value, which times log2 e are
# infinite, and an infinite value whose key's probability is 0
@pytest.mark.parametrize("ranges", [False, True])
@pytest.mark.parametrize("logits", [(-3e38, -3e38), (3e38, 3e38), (-3e38, -2.5e38), (-3e38, 1.0), (-1.5e38, -2.9e38),
                                    (-np.inf, 1.0), (-np.inf, -np.inf)])
def test_f32_logits_of_any_size(logits, ranges):
    nq, nk, hq, hkv, d = 20, 900, 2, 1, 64
    q, k, v, _ = _inputs(nq, nk, hq, hkv, d, seed=5)
    q.zero_(), k.zero_()
    q[..., 0], k[..., 0] = 1.0, logits[0]
    k[torch.arange(nk) % 3 == 1, :, 0] = logits[1]
    k[600:, :, 0] = max(logits)  # the last ranges hold one value alone
    pos = torch.arange(nq) * 45 + 44
    want, mass, size = _f64(q, k, v, pos, 1.0)
    got, whole = _attend_in_guards(*(t.to(DEV) for t in (q, k, v, pos)), 1.0, ranges)
    assert whole
    if max(logits) == -np.inf:  # no key has a weight: NaN, as the softmax is
        assert bool(torch.isnan(got).all())
        return
    assert np.all(np.abs(got.numpy() - want) <= _f32_bound(mass, 0.0, d, nk, 1.0))
    if logits == (-3e38, 1.0):
        # seen by all rows, at a probability of 0 of those that see a key past the first ranges
        k[:128, :, 0], v[0, 0, 3] = logits[0], float("inf")
        got, _ = _attend_in_guards(*(t.to(DEV) for t in (q, k, v, pos)), 1.0, ranges)
        assert bool(torch.isnan(got[3:, :, 3]).all()) and not bool(torch.isfinite(got[..., 3]).any())
        assert bool(torch.isfinite(got[..., 4:]).all())


# 16-bit rows around the 128-row tile, keys around the 32-key block and the
# four-block rings, ranges in which rows see nothing, and both merge widths;
# keys and queries in {-1, 0, 1} / 8, whose dot products are exact
@pytest.mark.parametrize("nq,nk,hq,hkv,d,dtype", [
    (1, 1, 1, 1, 128, torch.bfloat16), (1, 4097, 8, 8, 128, torch.bfloat16), (33, 1023, 4, 1, 64, torch.float16),
    (31, 700, 8, 2, 128, torch.float16), (129, 255, 1, 1, 64, torch.bfloat16), (64, 8191, 2, 2, 64, torch.bfloat16),
    (300, 3000, 16, 8, 128, torch.bfloat16), (17, 161, 5, 1, 128, torch.bfloat16),
])
def test_16_bit_matches_float64(nq, nk, hq, hkv, d, dtype):
    g = torch.Generator().manual_seed(nq)
    q, k = ((torch.randint(-1, 2, (n, h, d), generator=g) / 8).to(dtype) for n, h in ((nq, hq), (nk, hkv)))
    v = torch.randn(nk, hkv, d, generator=g).to(dtype)
    pos = torch.randint(0, nk, (nq,), generator=g)
    pos[-1] = nk - 1
    want, mass, _ = _f64(q, k, v, pos, 1.0)
    got = blend_attention(q.to(DEV), k.to(DEV), v.to(DEV), pos.to(DEV), 1.0).float().cpu().numpy()
    # the probabilities, their sum's terms and the output are each rounded once
    u = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    assert np.all(np.abs(got - want) <= 3 * u * mass + 1e-6)


def test_ranges_agree_with_one_range_far_above_the_first_blocks_maximum():
    # logits that outgrow each range's first block (the online second pass),
    # in some ranges only
    nq, nk, hq, hkv, d = 40, 4000, 4, 1, 128
    g = torch.Generator().manual_seed(3)
    q = torch.ones(nq, hq, d).to(torch.bfloat16).to(DEV)
    k = (torch.randint(-1, 2, (nk, hkv, d), generator=g) / 8).to(torch.bfloat16)
    k[1500:1510] = 1.5
    k[3900] = 2.0
    v = torch.randn(nk, hkv, d, generator=g).to(torch.bfloat16).to(DEV)
    pos = (torch.arange(nq) * 100 + 99).to(DEV)
    k = k.to(DEV)
    got = blend_attention(q, k, v, pos, 1.0)
    out = torch.empty_like(got)
    rc = _native.load().cbk_blend_attention(
        q.data_ptr(), hq * d, pos.data_ptr(), nq, k.data_ptr(), hkv * d, v.data_ptr(), hkv * d, nk, hq, hkv, d,
        1.0, _native.DTYPE_CODES[torch.bfloat16], out.data_ptr(), hq * d, _native.stream_handle(DEV))
    _native.check(rc, "blend_attention")
    diff = (got.float() - out.float()).abs()
    assert torch.isfinite(got).all()
    # each side rounds probabilities and outputs once: 2 * 2 * 2^-8 of values up to 4.5
    assert float(diff.max()) <= 4 * 2.0 ** -8 * 4.5


@pytest.mark.parametrize("ranges", [False, True])
@pytest.mark.parametrize("where", ["first block", "before low logits", "one range", "every range", "all"])
@pytest.mark.parametrize("dtype,d", [(torch.float16, 128), (torch.float16, 64), (torch.bfloat16, 128)])
def test_16_bit_first_blocks_of_minus_infinity(dtype, d, where, ranges):
    # rows whose logits in a range's first 32 keys are all -inf: in float16 a
    # finite dot product below -65504 (heads of zeros beside them, in the same
    # tiles), in bfloat16 a key of -inf
    nq, nk, hq, hkv = 40, 4000, 4, 1
    g = torch.Generator().manual_seed(6)
    q = torch.ones(nq, hq, d)
    k = torch.randint(-1, 2, (nk, hkv, d), generator=g) / 8
    k[torch.arange(nk) % 100 == 99] = 0.0625  # some keys far above the others
    if where == "before low logits":  # 2^-184 and less against a reference of 0
        k[:], k[torch.arange(nk) % 100 == 99] = -2.0, -2.0 + 0.0625
    value = -1024.0 if dtype == torch.float16 else -float("inf")
    if dtype == torch.float16:
        q[:, 1::2] = 0
    splits = _native.load().cbk_blend_attention_workspace_bytes(
        nq, nk, hq, hkv, d, _native.DTYPE_CODES[dtype]) // (nq * hq * (8 + 4 * d))
    assert splits > 8
    blocks = {"first block": [0], "before low logits": [0], "one range": [125 * 20 // splits], "all": range(125),
              "every range": [125 * s // splits for s in range(splits)]}[where]
    for b in blocks:
        k[32 * b:32 * b + 32] = value
    q, k, v = q.to(dtype), k.to(dtype), torch.randn(nk, hkv, d, generator=g).to(dtype)
    pos = torch.arange(nk - nq, nk)
    want, mass, _ = _f64(q, k.clamp(min=-1024.0), v, pos, 1.0)
    if where == "all":  # no key has a weight: zero
        rows = (q[..., 0] != 0).numpy()
        want[rows], mass[rows] = 0, 0
    print(f"{dtype} d={d} {where} ranges={ranges}", flush=True)
    got, whole = _attend_in_guards(*(t.to(DEV) for t in (q, k, v, pos)), 1.0, ranges)
    assert whole
    u = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    close = np.abs(got.float().numpy() - want) <= 3 * u * mass + 1e-6
    assert np.all(close)


@pytest.mark.parametrize("dtype,d,share", [(torch.bfloat16, 128, 0.01), (torch.bfloat16, 64, 0.01),
                                           (torch.float16, 128, 0.08)])
def test_16_bit_ranges_round_the_probabilities_of_one_range(dtype, d, share):
    # one reference per row for all ranges: the same probabilities, and sums
    # that differ in their order alone, by about sqrt(nk) 2^-24 of sum p |v|,
    # which is about sqrt(nk) |out| here: nk 2^-24 |out| = 1.8e-4 |out|. That
    # moves an output where it crosses a rounding boundary: 1.8e-4 / 2^-8 =
    # 4.6% of them at the most in bfloat16 and a fifth of that with errors of
    # either sign; 8 times as many in float16. With a reference of its own per
    # range the roundings themselves differ, and 42 to 46% of the outputs
    nq, nk, hq, hkv = 150, 3000, 8, 2
    q, k, v, pos = (t.to(DEV) for t in _inputs(nq, nk, hq, hkv, d, dtype, seed=11))
    k[0] *= 3  # a first block above the others, as prompts have
    a, _ = _attend_in_guards(q, k, v, pos, d ** -0.5, True)
    b, _ = _attend_in_guards(q, k, v, pos, d ** -0.5, False)
    differ = float((a != b).float().mean())
    print(f"share of outputs that differ {differ:.5f}", flush=True)
    assert differ <= share


# short contexts and full row tiles take one range (several were slower), long
# contexts of few rows as many as fill the chip
@pytest.mark.parametrize("nq,nk,hq,hkv,d,least,most", [
    (64, 256, 32, 8, 128, 1, 1), (256, 256, 8, 2, 64, 1, 1), (900, 1000, 32, 8, 128, 1, 1),
    (2000, 4000, 32, 8, 128, 1, 1), (7000, 32767, 32, 4, 128, 1, 1), (1000, 4000, 32, 8, 128, 2, 4),
    (1, 32767, 8, 8, 128, 8, 32), (180, 8191, 32, 8, 64, 6, 16), (1, 255, 1, 1, 64, 1, 1), (1, 255, 8, 8, 128, 1, 1),
])
def test_16_bit_ranges_where_they_pay(nq, nk, hq, hkv, d, least, most):
    code = _native.DTYPE_CODES[torch.bfloat16]
    nbytes = _native.load().cbk_blend_attention_workspace_bytes(nq, nk, hq, hkv, d, code)
    assert least <= max(1, nbytes // (nq * hq * (8 + 4 * d))) <= most


def test_no_memory_for_the_ranges(monkeypatch):
    # the call needs no scratch without them
    nq, nk, hq, hkv, d = 40, 3000, 8, 2, 128
    q, k, v, pos = _inputs(nq, nk, hq, hkv, d, torch.bfloat16, seed=8)
    q, k, v, pos = (t.to(DEV) for t in (q, k, v, pos))
    want = blend_attention(q, k, v, pos, d ** -0.5)
    empty = torch.empty

    def full(*args, **kw):
        if kw.get("dtype") == torch.uint8:
            raise torch.cuda.OutOfMemoryError("out of memory")
        return empty(*args, **kw)

    monkeypatch.setattr(torch, "empty", full)
    got = blend_attention(q, k, v, pos, d ** -0.5)
    # probabilities rounded against another reference, and the output: 2^-8 each, of values up to 4.5
    assert float((got.float() - want.float()).abs().max()) <= 4 * 2.0 ** -8 * 4.5
