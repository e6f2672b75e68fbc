"""Which sums of products a plan hands to the matrix cores beyond the aligned half widths (no GPU)."""

from __future__ import annotations

import numpy as np
import pytest

from limn_amd.seam import Node, Op, Tensor, bfloat16, custom, float32, grad, lower_all, realized, schedule, topological
from limn_amd.seam import device as limn_device

emit = pytest.importorskip("limn_amd.hip.emit")

rng = np.random.default_rng(5)


@pytest.fixture(autouse=True)
def on_numpy():
    limn_device.set_device("numpy")
    yield


def lowered(sinks: list[Tensor]):
    nodes = [t.node for t in sinks]
    order = topological(nodes)
    return lower_all(nodes, order, schedule(nodes, order)), {realized(s) for s in nodes}


def float32_layer(train: bool, act) -> tuple[list, list]:
    """A float32 Linear, `act`, Linear: the plan's roles for its sums, forward only or trained."""
    x = Tensor(rng.standard_normal((2048, 256)).astype(np.float32), requires_grad=True)
    w1, w2 = (Tensor(rng.standard_normal(s).astype(np.float32), requires_grad=True) for s in ((256, 128), (128, 256)))
    y = act(x @ w1) @ w2
    sinks = [y, *grad((y * y).sum(), [x, w1, w2])] if train else [y]
    nests, kept = lowered(sinks)
    prog = emit.plan_program(nests, kept, set())
    return nests, [p.contraction is not None for n, p in zip(nests, prog.plans) if n.kernel.ast.op is Op.SUM]


def test_float32_sums_a_mask_reads_keep_their_order():
    """A trained relu compares the first layer's sums to route gradients, so they stay on the general
    reduce kernels; every other product goes to the matrix cores. Without a backward, or with an
    activation that compares nothing, they all do."""
    assert float32_layer(True, lambda h: h.relu())[1].count(False) == 1
    assert all(float32_layer(False, lambda h: h.relu())[1])
    assert all(float32_layer(False, lambda h: h.minimum(1.0))[1])
    assert all(float32_layer(True, lambda h: h * h)[1])
    assert not float32_layer(False, lambda h: (h > 0).where(h * 2.0, h))[1][0]


def test_a_mask_reaches_back_through_attention():
    """The sums behind a CUSTOM call whose result a mask reads keep their order too."""
    q = Tensor(rng.standard_normal((4, 512, 64)).astype(np.float32))
    w = Tensor(rng.standard_normal((64, 64)).astype(np.float32))
    o, _ = custom("sdpa", ((q @ w).node, q.node, q.node), (True, 0.125), ((float32, (4, 512, 64)), (float32, (4, 512, 1))))
    att = Tensor.from_node(o)
    for picked, ordered in (((att > 0).where(att * 2.0, att), True), (att * 2.0, False)):
        sinks = [picked.node]
        order = topological(sinks)
        nests = [n for n in lower_all(sinks, order, schedule(sinks, order))]
        sums = [n for n in nests if n.kernel.ast.op is Op.SUM]
        assert len(sums) == 1 and (realized(sums[0].kernel.target) in emit.deciding(nests)) is ordered


@pytest.mark.parametrize("M,K,N,cores", [(513, 515, 517, True), (640, 1024, 129, True), (1023, 1031, 63, False), (300, 301, 303, False)], ids=str)
def test_unaligned_half_width_sums(M, K, N, cores):
    """Odd widths go to the copying contraction from 2^26 products, 64 of each side."""
    a, b = (Tensor(rng.standard_normal(s).astype(np.float32), dtype=bfloat16) for s in ((M, K), (K, N)))
    nests, kept = lowered([a @ b])
    (con,) = [p.contraction for n, p in zip(nests, emit.plan_program(nests, kept, set()).plans) if n.kernel.ast.op is Op.SUM]
    assert (con is not None) == cores
    assert con is None or not emit.takes_matmul(con)


# (layout, M, N, K): each general form on both sides of its line; n is x @ w^T, w x @ w, g x^T @ y
@pytest.mark.parametrize("layout,M,N,K,cores", [
    ("g", 10, 784, 4096, False), ("g", 64, 512, 4096, True), ("g", 24, 24, 26080, False), ("g", 256, 256, 1024, True), ("g", 64, 64, 4096, False),
    ("w", 2, 4096, 4096, False), ("w", 16, 4096, 4096, True), ("w", 64, 512, 512, False), ("w", 256, 256, 256, True), ("w", 2048, 2048, 2, False),
    ("n", 16, 16, 65536, False), ("n", 24, 24, 26080, False), ("n", 512, 512, 512, True), ("n", 64, 512, 512, True), ("n", 300, 300, 784, True),
], ids=str)
def test_float32_sums_go_where_they_are_faster(layout, M, N, K, cores):
    """Narrow sums, above all over a long k, stay on the general reduce kernels: measured, us, general /
    contract: g 10 x 784 x 4096 10.4/18.0, 24 x 24 x 26080 8.8/44, 64 x 64 x 4096 7.3/16.8; w 2 x 4096 x 4096
    20.3/29.7, 16 x 4096 x 4096 76/33, 64 x 512 x 512 7.3/9.1, 2048 x 2048 x 2 8.0/11.6; n 16 x 16 x 65536 7.7/113."""
    def operand(*shape):
        return Tensor.from_node(Node(Op.BUFFER, (), float32, shape, None))

    if layout == "g":
        out = operand(K, M).transpose() @ operand(K, N)
    else:
        out = operand(M, K) @ (operand(K, N) if layout == "w" else operand(N, K).transpose())
    nests, kept = lowered([out])
    (plan,) = [p for n, p in zip(nests, emit.plan_program(nests, kept, set()).plans) if n.kernel.ast.op is Op.SUM]
    assert (plan.contraction is not None) == cores


def test_a_declined_sum_keeps_its_epilogue_nests():
    """A narrow sum that stays general runs its bias and relu readers as nests of their own."""
    x, w = (Tensor.from_node(Node(Op.BUFFER, (), float32, s, None)) for s in ((65536, 24), (65536, 24)))
    nests, kept = lowered([(x.transpose() @ w).relu()])
    prog = emit.plan_program(nests, kept, set())
    assert not prog.pairs and all(p.contraction is None for p in prog.plans)


class Lib:
    """liblimn_hip.so's queries; its contraction entry records its arguments instead of running."""

    def __init__(self):
        self.calls = []

    def __getattr__(self, name):
        return getattr(emit.runtime.kernels(), name)

    def limn_hip_contract(self, *args):
        self.calls.append(args)
        return 0


def test_a_plans_contractions_share_one_workspace():
    """An odd-width layer and its gradients: every product copies operands, and all copies take turns in
    one allocation of the largest's size."""
    class Buf:
        ptr = 0x1000

    class Dev:
        plan_kept = plan_custom_inputs = tape = None

        def __init__(self):
            self.lib, self.sizes = Lib(), []

        def _alloc(self, nbytes):
            self.sizes.append(nbytes)
            return Buf()

    x, w, dy = (Tensor.from_node(Node(Op.BUFFER, (), bfloat16, s, None)) for s in ((2051, 515), (515, 517), (2051, 517)))
    nests, _ = lowered([x @ w, dy @ w.transpose(), x.transpose() @ dy])
    dev = Dev()
    runners = emit.nest_runners(dev, nests)
    assert len(runners) == 3
    for run, nest in zip(runners, nests):
        run([Buf()] * len(nest.kernel.inputs), [Buf()])
    needs = [args[-2] for args in dev.lib.calls]
    assert len(needs) == 3 and min(needs) > 0 and dev.sizes == [max(needs)]


def test_a_contraction_of_huge_copies_stays_general():
    """Copies past WORKSPACE_CAP: a bf16 product whose operands are 16 GB of odd rows each."""
    a, b = (Tensor.from_node(Node(Op.BUFFER, (), bfloat16, s, None)) for s in ((16, 257, 2000001), (16, 2000001, 255)))
    nests, kept = lowered([a @ b])
    (plan,) = [p for n, p in zip(nests, emit.plan_program(nests, kept, set()).plans) if n.kernel.ast.op is Op.SUM]
    assert plan.contraction is None
