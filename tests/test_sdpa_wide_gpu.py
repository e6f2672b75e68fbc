"""Float32-arithmetic attention on matrix cores (csrc/sdpa_wide.h), through the C ABI on the GPU.

Tolerance: every product, addition and exponential is float32 (half widths round once at the store);
against float64 over a few thousand keys the parts of a sum are at most 2e-6 of its terms' size, the
half widths' stores 2^-11 and 2^-8 of the value.
"""

from __future__ import annotations

import numpy as np
import pytest

from limn_amd.hip import runtime

pytestmark = pytest.mark.gpu

CODE = {"float32": 1, "float16": 2, "bfloat16": 3}
ROUND = {"float32": 0.0, "float16": 2.0**-10, "bfloat16": 2.0**-7}


def stored(x, dtype):
    from limn_amd.dtypes import from_storage, to_storage
    from limn_amd import seam

    t = getattr(seam, dtype)
    bits = to_storage(np.ascontiguousarray(x, dtype=np.float32), t)
    return bits, from_storage(bits.view(np.uint8), t, x.shape).astype(np.float64)


def run(dev, dtype, q, k, v, do, mask, causal, scale):
    """(out, lse, dq, dk, dv) of the device, as float64 values."""
    from limn_amd.dtypes import from_storage
    from limn_amd import seam

    t = getattr(seam, dtype)
    B, tq, hd = q.shape
    tk, hv = v.shape[1:]
    bufs = {}
    for name, x in (("q", q), ("k", k), ("v", v), ("do", do), ("mask", mask)):
        if x is not None:
            bits = stored(x, dtype)[0]
            bufs[name] = dev.alloc(bits.nbytes)
            dev.copyin(bufs[name], bits)
    size = t.itemsize
    out, lse = dev.alloc(B * tq * hv * size), dev.alloc(B * tq * 4)
    dq, dk, dv = dev.alloc(B * tq * hd * size), dev.alloc(B * tk * hd * size), dev.alloc(B * tk * hv * size)
    m = bufs["mask"].ptr if mask is not None else None
    sizes = (CODE[dtype], B, tq, tk, hd, hv, int(causal), scale, None)
    runtime.check_limn(dev.lib.limn_hip_sdpa_fwd(bufs["q"].ptr, bufs["k"].ptr, bufs["v"].ptr, m, out.ptr, lse.ptr, *sizes))
    o = from_storage(dev.copyout(out), t, (B, tq, hv)).astype(np.float64)
    with np.errstate(invalid="ignore"):
        delta = (stored(do, dtype)[1] * o).sum(-1).astype(np.float32)
    d = dev.alloc(delta.nbytes)
    dev.copyin(d, delta)
    args = (bufs["q"].ptr, bufs["k"].ptr, bufs["v"].ptr, bufs["do"].ptr, lse.ptr, d.ptr, m)
    runtime.check_limn(dev.lib.limn_hip_sdpa_bwd_q(*args, dq.ptr, *sizes))
    runtime.check_limn(dev.lib.limn_hip_sdpa_bwd_kv(*args, dk.ptr, dv.ptr, *sizes))
    dev.finish()
    back = lambda b, shape: from_storage(dev.copyout(b), t, shape).astype(np.float64)
    return o, dev.copyout(lse).view(np.float32).reshape(B, tq), back(dq, (B, tq, hd)), back(dk, (B, tk, hd)), back(dv, (B, tk, hv))


def exact(dtype, q, k, v, do, mask, causal, scale):
    q, k, v, do = (stored(x, dtype)[1] for x in (q, k, v, do))
    s = q @ k.swapaxes(1, 2) * scale
    if causal:
        s = np.where(np.tril(np.ones(s.shape[1:], bool)), s, -np.inf)
    if mask is not None:
        s = np.where(mask[:, None, :] != 0, s, -np.inf)
    top = s.max(-1, keepdims=True)
    p = np.exp(s - top)
    total = p.sum(-1, keepdims=True)
    p /= total
    o = p @ v
    dp = do @ v.swapaxes(1, 2)
    ds = p * (dp - (do * o).sum(-1, keepdims=True)) * scale
    return o, (top + np.log(total))[..., 0], ds @ k, ds.swapaxes(1, 2) @ q, p.swapaxes(1, 2) @ do


# (batch, t_q, t_k, hd, hd_v, causal, masked): block and tile edges (32), one to many tiles a wave, padded
# dims at each width (32, 64, 96, 128), unequal dims, paired causal blocks (512 units), a wave a block (8192 blocks)
CASES = [
    (33, 32, 32, 32, 32, True, False), (5, 65, 65, 20, 28, True, True), (40, 33, 200, 64, 64, False, True), (9, 300, 129, 80, 64, False, False),
    (70, 127, 127, 128, 128, True, False), (6, 400, 400, 96, 96, True, True), (130, 50, 34, 16, 4, False, False), (64, 513, 513, 32, 32, True, False),
    (4100, 64, 64, 32, 32, True, False), (8200, 32, 40, 4, 8, False, True),
]


@pytest.mark.parametrize("dtype", list(CODE))
@pytest.mark.parametrize("case", CASES, ids=str)
def test_matches_float64(hipdev, case, dtype):
    B, tq, tk, hd, hv, causal, masked = case
    rng = np.random.default_rng(tq + hd)
    q, k, v, do = (rng.standard_normal(s) for s in ((B, tq, hd), (B, tk, hd), (B, tk, hv), (B, tq, hv)))
    mask = (rng.random((B, tk)) < 0.7).astype(np.float64) if masked else None
    if masked:
        mask[:, 0] = 1
    narrow = dtype != "float32" and hd == hv and hd in (64, 128)  # the 16-bit family's backward
    for scale in (hd**-0.5,) if narrow else (hd**-0.5, -0.3):
        got, want = run(hipdev, dtype, q, k, v, do, mask, causal, scale), exact(dtype, q, k, v, do, mask, causal, scale)
        for name, g, w in zip(("out", "lse", "dq", "dk", "dv"), got, want):
            # delta is summed from the rounded output: its rounding reaches dq and dk at the size of the row
            rel = 1e-5 + (ROUND[dtype] if name != "lse" else 0.0)
            np.testing.assert_allclose(g, w, rtol=rel, atol=rel * max(1.0, np.abs(w).max()), err_msg=name)


# one streamed tile (a wave a block at any number of blocks), two and three (from 2048 blocks), and the calls of
# few blocks beside them that stay on the rows kernels
SHORT_CASES = [(700, 96, 96, 32, 32, True, False), (1030, 64, 40, 80, 64, False, True), (140, 32, 100, 128, 128, False, False),
               (300, 100, 32, 64, 64, False, True), (129, 32, 32, 16, 16, True, False), (40, 32, 32, 128, 96, True, True), (16, 64, 64, 128, 128, True, False)]


@pytest.mark.parametrize("dtype", ["float32", "float16"])
@pytest.mark.parametrize("case", SHORT_CASES, ids=str)
def test_short_streams_match_float64(hipdev, case, dtype):
    test_matches_float64(hipdev, case, dtype)


def test_hidden_keys_keep_their_garbage_to_themselves(hipdev):
    """Masked keys may hold NaN or infinities: no live row or key sees them."""
    B, t, d = 8, 150, 64
    rng = np.random.default_rng(0)
    q, k, v, do = (rng.standard_normal((B, t, d)) for _ in range(4))
    mask = np.ones((B, t))
    mask[:, 100:] = 0
    clean = run(hipdev, "float32", q, k, v, do, mask, False, 0.125)
    k[:, 100:], v[:, 100:] = np.nan, np.inf
    got = run(hipdev, "float32", q, k, v, do, mask, False, 0.125)
    for g, c in zip(got[:3], clean[:3]):
        np.testing.assert_array_equal(g, c)
    for g, c in zip(got[3:], clean[3:]):
        np.testing.assert_array_equal(g[:, :100], c[:, :100])


@pytest.mark.parametrize("at", [3, 40, 95])
def test_a_causal_row_sees_no_later_infinity(hipdev, at):
    """An infinity in one value row and a NaN in one dO row: rows before (queries) and keys after (for dO)
    stay as they were, and the rows that do read it are not finite."""
    B, t, d = 12, 96, 32
    rng = np.random.default_rng(1)
    q, k, v, do = (rng.standard_normal((B, t, d)) for _ in range(4))
    clean = run(hipdev, "float32", q, k, v, do, None, True, 0.2)
    broken = v.copy()
    broken[:, at, 5] = np.inf
    got = run(hipdev, "float32", q, k, broken, do, None, True, 0.2)
    np.testing.assert_array_equal(got[0][:, :at], clean[0][:, :at])
    assert np.isposinf(got[0][:, at:, 5]).all()
    np.testing.assert_array_equal(np.delete(got[0], 5, axis=2), np.delete(clean[0], 5, axis=2))
    np.testing.assert_array_equal(got[2][:, :at], clean[2][:, :at])  # dq of the rows before it
    broken = do.copy()
    broken[:, at, 7] = np.nan
    got = run(hipdev, "float32", q, k, v, broken, None, True, 0.2)
    np.testing.assert_array_equal(got[4][:, at + 1 :], clean[4][:, at + 1 :])  # dv of keys its query does not see
    assert np.isnan(got[4][:, : at + 1, 7]).all()


def test_same_bits_twice(hipdev):
    rng = np.random.default_rng(2)
    x = [rng.standard_normal((64, 520, 32)) for _ in range(4)]
    a, b = (run(hipdev, "float32", *x, None, True, 0.2) for _ in range(2))
    for p, q in zip(a, b):
        np.testing.assert_array_equal(p, q)


# (batch, t_q, t_k, hd, hd_v, masked): query and key tile edges (128, 64), each padded width, unequal dims
SPLIT_CASES = [(20, 1, 64, 32, 32, False), (16, 129, 65, 16, 24, True), (3, 128, 63, 64, 40, True), (2, 130, 200, 96, 96, False),
               (2, 40, 129, 80, 80, True), (1, 7, 1, 128, 104, False), (5, 64, 512, 120, 120, True)]


@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
@pytest.mark.parametrize("case", SPLIT_CASES, ids=str)
def test_split_probabilities_match_float64(hipdev, case, dtype):
    """The non-causal half-width forward (csrc/sdpa_split.hip): one rounding at the store is all it adds."""
    B, tq, tk, hd, hv, masked = case
    rng = np.random.default_rng(tk)
    q, k, v, do = (rng.standard_normal(s) for s in ((B, tq, hd), (B, tk, hd), (B, tk, hv), (B, tq, hv)))
    mask = (rng.random((B, tk)) < 0.6).astype(np.float64) if masked else None
    if masked:
        mask[:, -1] = 1
    want = exact(dtype, q, k, v, do, mask, False, hd**-0.5)
    if masked:  # what a hidden key holds reaches nothing
        k, v = np.where(mask[..., None] != 0, k, np.inf), np.where(mask[..., None] != 0, v, np.nan)
    got = run(hipdev, dtype, q, k, v, do, mask, False, hd**-0.5)
    rel = ROUND[dtype] / 2 + 1e-5  # half an ulp of the stored value
    np.testing.assert_allclose(got[0], want[0], rtol=rel, atol=1e-5)
    np.testing.assert_allclose(got[1], want[1], rtol=1e-5, atol=1e-5)
    if masked:
        mask[0] = 0  # a row with every key hidden: NaN, and lse -inf
        got = run(hipdev, dtype, q, k, v, do, mask, False, hd**-0.5)
        assert np.isnan(got[0][0]).all() and np.isneginf(got[1][0]).all() and np.isfinite(got[0][1:]).all()


@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
@pytest.mark.parametrize("case", [(16, 129, 65, 32, 24, True), (3, 128, 63, 64, 40, False), (2, 40, 200, 128, 104, True)], ids=str)
def test_split_probabilities_carry_an_infinity(hipdev, case, dtype):
    """An infinity in a live value row reaches its dim of every query with its sign, also at weights that
    16 bits hold exactly (no remainder) or round to zero; two that meet make NaN; other dims and other
    heads keep their bits."""
    B, tq, tk, hd, hv, masked = case
    rng = np.random.default_rng(tk)
    q, k, v, do = (rng.standard_normal(s) for s in ((B, tq, hd), (B, tk, hd), (B, tk, hv), (B, tq, hv)))
    q[0, 1] = 0  # every weight 1
    q[0, 2] = 8 * k[0, 0] / np.abs(k[0, 0]).max()  # most weights tiny
    scale = hd**-0.5
    mask = np.ones((B, tk)) if masked else None
    if masked:
        mask[:, 7:20] = 0
    clean = run(hipdev, dtype, q, k, v, do, mask, False, scale)
    v[0, 40, 3], v[0, 41, 9], v[0, [5, 50], 17] = np.inf, -np.inf, [np.inf, -np.inf]
    got = run(hipdev, dtype, q, k, v, do, mask, False, scale)
    assert np.isposinf(got[0][0, :, 3]).all() and np.isneginf(got[0][0, :, 9]).all() and np.isnan(got[0][0, :, 17]).all()
    np.testing.assert_array_equal(np.delete(got[0][0], [3, 9, 17], axis=1), np.delete(clean[0][0], [3, 9, 17], axis=1))
    np.testing.assert_array_equal(got[0][1:], clean[0][1:])
    np.testing.assert_array_equal(got[1], clean[1])


def weighed(dtype, q, k, v, scale):
    """The forward's output in float64; the sum of the sizes of its terms; the largest exponent (log2) of a weight."""
    q, k, v = (stored(x, dtype)[1] for x in (q, k, v))
    s = q @ k.swapaxes(1, 2) * scale
    s -= s.max(-1, keepdims=True)
    p = np.exp(s)
    p /= p.sum(-1, keepdims=True)
    return p @ v, p @ np.abs(v), -s.min() / np.log(2)


def forward(dev, dtype, q, k, v, scale):
    """(out, lse) of the device's forward."""
    from limn_amd.dtypes import from_storage
    from limn_amd import seam

    t = getattr(seam, dtype)
    B, tq, hd = q.shape
    tk, hv = v.shape[1:]
    bufs = []
    for x in (q, k, v):
        bits = stored(x, dtype)[0]
        bufs.append(dev.alloc(bits.nbytes))
        dev.copyin(bufs[-1], bits)
    out, lse = dev.alloc(B * tq * hv * t.itemsize), dev.alloc(B * tq * 4)
    runtime.check_limn(dev.lib.limn_hip_sdpa_fwd(*(b.ptr for b in bufs), None, out.ptr, lse.ptr, CODE[dtype], B, tq, tk, hd, hv, 0, scale, None))
    dev.finish()
    return from_storage(dev.copyout(out), t, (B, tq, hv)).astype(np.float64), dev.copyout(lse).view(np.float32).reshape(B, tq)


def assert_float32_weights(got, want, size, far, dtype):
    """A term of the sum in float32: its weight's exponent t = c s - c m carries the rounding of c (|t| 2^-24
    of it) and its own, its score a few roundings, its product and additions a few more, (10 + 2 |t|) 2^-24
    of the term in all. The store rounds once, in float16 to no less than 2^-25."""
    step = ROUND[dtype] / 2
    bound = step * np.abs(want) + (10 + 2 * far) * 2.0**-24 * size + (2.0**-25 if dtype == "float16" else 0.0)
    worst = (np.abs(got - want) / bound).max()
    assert worst <= 1, f"{worst:.2f} times the bound"


@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
@pytest.mark.parametrize("hd,hv", [(32, 32), (64, 40), (80, 80), (120, 120)], ids=str)
def test_split_probabilities_hold_float32_weights(hipdev, hd, hv, dtype):
    """Outputs whose terms cancel to 2^-15 of their spread, where the store's own rounding (2^-8 of them) is
    under float32's: the terms' errors are then a few independent roundings, together some 2^-22.5 of
    the spread in root mean square. Weights of 16 bits leave 2^-19.5."""
    B, tq, tk = 3840 // hv, 1024, 48
    rng = np.random.default_rng(hd)
    q, k, v = (rng.standard_normal(s) for s in ((B, tq, hd), (B, tk, hd), (B, tk, hv)))
    v *= 256
    got = forward(hipdev, dtype, q, k, v, hd**-0.5)[0]
    q, k, v = (stored(x, dtype)[1] for x in (q, k, v))
    p = np.exp(q @ k.swapaxes(1, 2) * hd**-0.5)
    p /= p.sum(-1, keepdims=True)
    want, spread = p @ v, np.sqrt((p * p) @ (v * v))
    near = np.abs(want) < 2.0**-15 * spread
    assert near.sum() > 40
    assert np.sqrt(np.mean(((got - want)[near] / spread[near]) ** 2)) < 2.0**-21


@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
@pytest.mark.parametrize("gap", [10, 14, 17, 20, 23])
@pytest.mark.parametrize("case", [(16, 3, 1021, 32, 32), (2, 40, 4096, 80, 80), (2, 40, 1021, 96, 120)], ids=str)
def test_split_probabilities_keep_small_weights(hipdev, case, gap, dtype):
    """One key of weight near 1 and value zero among keys `gap` nats below it: the output is theirs alone,
    and lse counts them too."""
    B, tq, tk, hd, hv = case
    rng = np.random.default_rng(tk + gap)
    q, k = np.ones((B, tq, hd)), rng.standard_normal((B, tk, hd))
    v = np.abs(rng.standard_normal((B, tk, hv))) * 1000
    k[:, 300], v[:, 300] = gap * hd**-0.5, 0  # in a later tile than the first: the reference point moves to it
    want, size, far = weighed(dtype, q, k, v, hd**-0.5)
    assert_float32_weights(forward(hipdev, dtype, q, k, v, hd**-0.5)[0], want, size, far, dtype)


@pytest.mark.parametrize("dtype,size", [("float16", 2e3), ("float16", 1e4), ("bfloat16", 2e4), ("bfloat16", 3e6), ("bfloat16", 1e15)], ids=str)
@pytest.mark.parametrize("hd,hv", [(32, 32), (80, 80), (96, 120)], ids=str)
def test_split_probabilities_of_far_scores(hipdev, hd, hv, dtype, size):
    """Scores of 10^7 to 10^31: a row is its nearest key's value row (the others are further below it
    than its score's own rounding), and lse its score."""
    B, tq, tk = 16, 40, 200
    rng = np.random.default_rng(hd)
    q, k, v = (rng.standard_normal(s) for s in ((B, tq, hd), (B, tk, hd), (B, tk, hv)))
    q, k, v = (stored(x, dtype)[1] for x in (q * size, k * size, v))
    k[:, 150] = k[:, 20]  # an equal score in a later tile
    s = np.sort(q @ np.delete(k, 150, axis=1).swapaxes(1, 2), axis=-1) * hd**-0.5
    clear = s[..., -1] - s[..., -2] > 40 + np.abs(s[..., -1]) * hd * 2.0**-23
    assert clear.mean() > 0.9
    want, _, _ = weighed(dtype, q, k, v, hd**-0.5)
    out, lse = forward(hipdev, dtype, q, k, v, hd**-0.5)
    np.testing.assert_allclose(out[clear], want[clear], rtol=ROUND[dtype] / 2 + 1e-5, atol=1e-5)
    np.testing.assert_allclose(lse[clear], s[..., -1][clear], rtol=(hd + 2) * 2.0**-23)


@pytest.mark.parametrize("hd", [32, 80, 120])
def test_a_score_past_float32_stays_in_its_row(hipdev, hd):
    """Finite bfloat16 queries and keys whose score is infinite: NaN in that row, as exp(inf - inf) is, a
    weight of 0 where it is -inf, and every other row of the workgroup's second walk as without it."""
    B, tq, tk = 16, 40, 130
    rng = np.random.default_rng(hd)
    q, k, v = (rng.standard_normal(s) for s in ((B, tq, hd), (B, tk, hd), (B, tk, hd)))
    q[:, 5], q[:, 6], k[:, 70] = 1e20, -1e20, 1e20
    out, lse = forward(hipdev, "bfloat16", q, k, v, hd**-0.5)
    assert np.isnan(out[:, 5]).all() and np.isnan(lse[:, 5]).all()
    q, k, v = (stored(x, "bfloat16")[1] for x in (q, k, v))
    top = np.argmax(q @ k.swapaxes(1, 2), axis=-1)
    rest = np.delete(np.arange(tq), 5)
    sure = np.abs(q.sum(-1)) > 1  # rows whose score with key 70 is far from the others, whatever its rounding
    want = np.take_along_axis(v, top[..., None], 1)
    assert np.isfinite(out[:, rest]).all() and sure.mean() > 0.7
    np.testing.assert_array_equal(out[:, rest][(sure & (top == 70))[:, rest]], want[:, rest][(sure & (top == 70))[:, rest]])
    np.testing.assert_array_equal(out[:, 6], want[:, 6])


@pytest.mark.parametrize("hd", [24, 32, 48, 80, 96, 128])
def test_a_far_score_keeps_its_whole_weight(hipdev, hd):
    """Queries in line with one key, its score thousands above the others': a weight of exactly 1, whatever
    the score's rounding, so dV is the plain sum of those queries' dO, and the output the key's row."""
    B, tq, tk = 32, 200, 70
    rng = np.random.default_rng(hd)
    k, v, do = (rng.standard_normal(s).astype(np.float32) for s in ((B, tk, hd), (B, tk, hd), (B, tq, hd)))
    k *= (8 / np.linalg.norm(k, axis=-1, keepdims=True)).astype(np.float32)
    pick = rng.integers(0, tk, (B, tq))
    q = 1234.5 * np.take_along_axis(k, pick[..., None], 1)
    out, lse, _, _, dv = run(hipdev, "float32", q, k, v, do, None, False, 0.3)
    np.testing.assert_array_equal(out, np.take_along_axis(v, pick[..., None], 1))
    hot = (pick[..., None] == np.arange(tk)).astype(np.float64).swapaxes(1, 2)
    assert (np.abs(dv - hot @ do) <= 16 * 2.0**-24 * (hot @ np.abs(do))).all()  # a key has some 3 queries, 10 at most
