"""limn_hip_contract, the contraction of float32 and of unaligned half widths, through the C ABI on the GPU and through plans of nests.

Tolerance in float32: a product and an addition of a sum each round once (2^-24 of the value), a running
total is at most 64 products long, then the 64-long totals and the k slices are added, so the error
of a cell is under (64 + K / 64 + slices + 3) 2^-24 times its sum of |a b| (and the terms').
"""

from __future__ import annotations

import numpy as np
import pytest

from limn_amd.hip import runtime
from limn_amd.seam import Tensor, float32, use_device

pytestmark = pytest.mark.gpu
F32 = 1


def upload(dev, x: np.ndarray, offset: int = 0):
    """x in a device buffer, `offset` floats past its start; (buffer, pointer)."""
    flat = np.concatenate([np.full(offset, np.nan, np.float32), np.ascontiguousarray(x, dtype=np.float32).reshape(-1)])
    buf = dev.alloc(flat.nbytes)
    dev.copyin(buf, flat)
    return buf, buf.ptr + 4 * offset


# tile edges (64, 128), stage edges (32), k tails, one row or column, a split k, a shape of 128 x 128 tiles
SHAPES = [(1, 1, 1), (64, 64, 32), (65, 63, 33), (130, 127, 31), (33, 200, 300), (7, 1030, 1), (40, 24, 4100), (256, 256, 1024), (2944, 2950, 36)]


@pytest.mark.parametrize("a_kcontig", [True, False], ids=["a-k", "a-m"])
@pytest.mark.parametrize("b_kcontig", [True, False], ids=["b-k", "b-n"])
@pytest.mark.parametrize("M,N,K", SHAPES, ids=str)
def test_contract_layouts(hipdev, a_kcontig, b_kcontig, M, N, K):
    rng = np.random.default_rng(M + N + K)
    batch = 2 if M < 1000 else 1
    a, b = rng.standard_normal((batch, M, K)).astype(np.float32), rng.standard_normal((batch, K, N)).astype(np.float32)
    bias, res = rng.standard_normal(N).astype(np.float32), rng.standard_normal((batch, M, N)).astype(np.float32)
    odd = (M + N + K) % 2  # half the shapes start one float past a 16-byte boundary
    keep_a, pa = upload(hipdev, a if a_kcontig else a.swapaxes(1, 2), odd)
    keep_b, pb = upload(hipdev, b.swapaxes(1, 2) if b_kcontig else b, odd)
    keep_bias, pbias = upload(hipdev, bias)
    keep_res, pres = upload(hipdev, res, odd)
    (a_m, a_k), (b_k, b_n) = ((K, 1) if a_kcontig else (1, M)), ((1, K) if b_kcontig else (N, 1))
    lib = hipdev.lib
    need = lib.limn_hip_contract_workspace(F32, batch, M, N, K, M * K, a_m, a_k, K * N, b_k, b_n, 0)
    ws = hipdev.alloc(max(need, 4))
    total = a.astype(np.float64) @ b.astype(np.float64)
    size = np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64)
    for turned, relu, terms, room in ((False, 0, True, need), (False, 1, False, 0), (True, 0, False, need)):
        guard = 5  # cells past the output that must stay as they were
        keep_c, pc = upload(hipdev, np.full(batch * M * N + guard, 7.0), odd)
        c_m, c_n = (1, M) if turned else (N, 1)
        runtime.check_limn(lib.limn_hip_contract(pa, pb, pc, F32, batch, M, N, K, M * K, a_m, a_k, K * N, b_k, b_n, M * N, c_m, c_n, relu,
                                                 pbias if terms else None, F32, 1, pres if terms else None, M * N, N, 1, ws.ptr, room, None))
        hipdev.finish()
        got = hipdev.copyout(keep_c).view(np.float32)[odd:]
        assert (got[batch * M * N :] == 7.0).all()
        got = got[: batch * M * N].reshape((batch, N, M) if turned else (batch, M, N))
        got = got.swapaxes(1, 2) if turned else got
        want, bound = np.maximum(total, 0.0) if relu else total, size
        if terms:
            want, bound = res + (want + bias), size + np.abs(bias) + np.abs(res)
        slices = 1 if not room else -(-need // (4 * batch * M * N))
        assert (np.abs(got - want) <= (min(K, 64) + K / 64 + slices + 3) * 2.0**-24 * bound).all()


def test_contract_keeps_infinities_and_nans_to_their_rows(hipdev):
    M, N, K = 100, 70, 37  # a k tail: the padding must not meet the infinities
    rng = np.random.default_rng(0)
    a, b = rng.standard_normal((M, K)).astype(np.float32), np.abs(rng.standard_normal((K, N))).astype(np.float32)
    a[3, 36], a[50, 0] = np.inf, np.nan
    keep_a, pa = upload(hipdev, a)
    keep_b, pb = upload(hipdev, b)
    c = hipdev.alloc(4 * M * N)
    runtime.check_limn(hipdev.lib.limn_hip_contract(pa, pb, c.ptr, F32, 1, M, N, K, 0, K, 1, 0, N, 1, 0, N, 1, 0, None, F32, 1, None, 0, 0, 0, None, 0, None))
    hipdev.finish()
    got = hipdev.copyout(c).view(np.float32).reshape(M, N)
    assert np.isposinf(got[3]).all() and np.isnan(got[50]).all()
    assert np.isfinite(np.delete(got, (3, 50), axis=0)).all()


def test_contract_takes_overlapping_and_broadcast_rows(hipdev):
    """A sliding window (a[m + k]: both strides 1) and a left operand shared by the batch."""
    M, N, K, batch = 77, 33, 45, 3
    rng = np.random.default_rng(1)
    x, b = rng.standard_normal(M + K - 1).astype(np.float32), rng.standard_normal((batch, K, N)).astype(np.float32)
    keep_a, pa = upload(hipdev, x)
    keep_b, pb = upload(hipdev, b)
    c = hipdev.alloc(4 * batch * M * N)
    runtime.check_limn(hipdev.lib.limn_hip_contract(pa, pb, c.ptr, F32, batch, M, N, K, 0, 1, 1, K * N, N, 1, M * N, N, 1, 0, None, F32, 1, None, 0, 0, 0, None, 0, None))
    hipdev.finish()
    a = np.lib.stride_tricks.sliding_window_view(x, K).astype(np.float64)
    got = hipdev.copyout(c).view(np.float32).reshape(batch, M, N)
    assert (np.abs(got - a @ b) <= (K + 3) * 2.0**-24 * (np.abs(a) @ np.abs(b))).all()


def test_contract_refuses_what_it_cannot_run(hipdev):
    lib, p = hipdev.lib, hipdev.alloc(64).ptr

    def call(dtype=F32, K=4, a_m=4, a_k=1, bias_dtype=F32, c=p, ws=0):
        return lib.limn_hip_contract(p, p, c, dtype, 1, 4, 4, K, 0, a_m, a_k, 0, 4, 1, 0, 4, 1, 0, p, bias_dtype, 1, None, 0, 0, 0, None, ws, None)

    assert [call(dtype=0), call(a_m=8, a_k=2), call(a_m=1 << 30)] == [2, 2, 2]
    assert [call(K=0), call(bias_dtype=3), call(c=p + 2), call(ws=-1), call(dtype=3, bias_dtype=3)] == [1, 1, 1, 1, 1]


# (a-k, b-k): each layout at one element, odd sizes, a k of whole 8s beside ragged rows, k tails about a
# stage (64), rows wider than a tile, a split k
HALF_SHAPES = [(1, 1, 1), (7, 9, 64), (65, 63, 65), (130, 127, 136), (33, 257, 63), (40, 24, 4099), (300, 517, 129)]


@pytest.mark.parametrize("layout", [(1, 1), (1, 0), (0, 1), (0, 0)], ids=["kk", "kn", "mk", "mn"])
@pytest.mark.parametrize("M,N,K", HALF_SHAPES, ids=str)
def test_contract_half_widths_any_alignment(hipdev, layout, M, N, K):
    """Whole numbers up to 8 in float16: every product and float32 total is exact, so the result is the
    float64 one rounded to float16, then rounded again with the terms added (limn_hip_matmul_add's
    rule). The operands sit between NaNs, half of them off a 16-byte boundary."""
    rng = np.random.default_rng(M + N + K)
    half, batch, lib = 2, 2, hipdev.lib
    shift = [(M + K) % 2, (N // 8) % 2 * 3]

    def put(x, off):
        flat = np.concatenate([np.full(off, np.nan), x.reshape(-1), np.full(9, np.nan)]).astype(np.float16)
        buf = hipdev.alloc(flat.nbytes)
        hipdev.copyin(buf, flat)
        return buf, buf.ptr + 2 * off

    a, b = (rng.integers(-8, 9, (batch, *d)).astype(np.float64) for d in ((M, K), (K, N)))
    bias, res = rng.integers(-8, 9, N).astype(np.float64), rng.integers(-8, 9, (batch, M, N)).astype(np.float64)
    a[0, 0, 0] = np.inf  # stays in its row
    b[1, K - 1, N - 1] = np.nan  # and this in its column
    keep_a, pa = put(a if layout[0] else a.swapaxes(1, 2), shift[0])
    keep_b, pb = put(b.swapaxes(1, 2) if layout[1] else b, shift[1])
    keep_bias, pbias = put(bias, 1)
    keep_res, pres = put(res, 1)
    keep_c, pc = put(np.full(batch * M * N, 7.0), 1)
    (a_m, a_k), (b_k, b_n) = ((K, 1) if layout[0] else (1, M)), ((1, K) if layout[1] else (N, 1))
    sizes = (half, batch, M, N, K, M * K, a_m, a_k, K * N, b_k, b_n)
    shifted = (pa % 16 != 0) + 2 * (pb % 16 != 0)
    assert lib.limn_hip_contract_supported(*sizes, shifted)
    need = lib.limn_hip_contract_workspace(*sizes, shifted)
    ws = hipdev.alloc(max(need, 16))
    hipdev.copyin(ws, np.full(max(need, 16) // 4, np.nan, np.float32))
    call = (pa, pb, pc, *sizes, M * N, N, 1, 0, pbias, half, 1, pres, M * N, N, 1, ws.ptr)
    if need:
        assert lib.limn_hip_contract(*call, need - 1, None) == 1
    runtime.check_limn(lib.limn_hip_contract(*call, need, None))
    hipdev.finish()
    got = hipdev.copyout(keep_c).view(np.float16)
    assert np.isnan(got[1 + batch * M * N :]).all() and np.isnan(got[0])
    with np.errstate(invalid="ignore"):
        total = (a @ b).astype(np.float16).astype(np.float64)
        want = (res + (total + bias)).astype(np.float16)
    np.testing.assert_array_equal(got[1 : 1 + batch * M * N].reshape(batch, M, N), want)


@pytest.mark.parametrize("lead", [(512,), (4, 128)], ids=["rows", "batched"])
def test_a_float32_linear_and_its_gradients_on_matrix_cores(hipdev, lead):
    """x @ w^T + b and its gradients, over shapes past the size rule, against float64."""
    from limn_amd.seam import grad

    use_device(hipdev)
    rng = np.random.default_rng(2)
    x, w, b, dy = (rng.standard_normal(s).astype(np.float32) for s in (lead + (200,), (121, 200), (121,), lead + (121,)))
    X, W, B = (Tensor(t, requires_grad=True) for t in (x, w, b))
    y = X @ W.transpose() + B
    got = [t.numpy() for t in (y, *grad((y * Tensor(dy)).sum(), [X, W, B]))]
    x2, dy2 = x.reshape(-1, 200).astype(np.float64), dy.reshape(-1, 121).astype(np.float64)
    want = [x2 @ w.T + b, dy2 @ w, dy2.T @ x2, dy2.sum(0)]
    for g, e in zip(got, want):
        np.testing.assert_allclose(g.reshape(e.shape), e, rtol=1e-5, atol=1e-5 * np.sqrt(np.mean(e * e)) * 4)


# lane groups of 1, 8, 16, 32 and 64, chunks of 4, 2 and 1, ragged block edges, both block sizes, a batch, one operand twice
@pytest.mark.parametrize("lead,k,n", [((4100,), 32, 1030), ((700,), 64, 700), ((333,), 130, 1290), ((512,), 512, 512), ((257,), 1021, 515),
                                      ((300,), 784, 300), ((65,), 3000, 601), ((3, 130), 96, 530)], ids=str)
def test_blocks_of_ordered_sums_give_the_bits_of_one_cell_a_group(hipdev, monkeypatch, lead, k, n):
    """plan_tiled against the plan it replaces, forward sums that a comparison keeps off the matrix cores."""
    from limn_amd.hip import emit

    use_device(hipdev)
    rng = np.random.default_rng(k)
    x, w = Tensor(rng.standard_normal((*lead, k)).astype(np.float32)), Tensor(rng.standard_normal((n, k)).astype(np.float32))
    kinds = []
    blocks = emit.plan_tiled
    monkeypatch.setattr(emit, "plan_tiled", lambda *a: kinds.append(blocks(*a)) or kinds[-1])

    def run(b):
        hipdev.plans.clear()
        h = x @ b.transpose()
        out = (h > 0).where(h * 2.0, h)
        return [hipdev.copyout(buf) for buf in hipdev.execute([h.node, out.node])]

    got = [run(w)] + ([run(x)] if len(lead) == 1 else [])
    assert kinds[0] is not None and "tiled" in kinds[0].notes
    monkeypatch.setattr(emit, "plan_tiled", lambda *a: None)
    want = [run(w)] + ([run(x)] if len(lead) == 1 else [])
    hipdev.plans.clear()
    for g, e in zip(got, want):
        for a, b in zip(g, e):
            np.testing.assert_array_equal(a, b)
