"""The work a user of the hip device has it do, as cases that can be timed and checked.

Every case goes through what a program calls: limn's Tensor API on `set_device("hip")`, the step
captured once per configuration (`capture`) and called with the pass's buffers; the attention
forward of a server goes through the C ABI of liblimn_hip.so instead. Inputs are made on the GPU from a
seed; `exact` computes the same values in float64 with plain torch.

Kinds and their ranges (`draw` takes sizes over all of them, the listed cases are points in them):

- attention: bf16, f16 and f32, head dims 16 to 128, 32 to 4096 positions, causal or not, with and
  without a key mask, square and rectangular; trained (forward, dQ, dK, dV) or served (forward);
- matmul: one product with a relu after it, bf16, f16 and f32, 33 to 4096 a side, odd sizes too;
- mlp: two Linear layers, forward and backward, in float32 (limn's default type) or in bf16 over
  float32 masters, 16 to 16384 rows;
- norm: row softmax then LayerNorm, float32;
- adamw: one optimizer step over the parameters of a transformer block, updated in place;
- gpt: forward and backward of the byte-level GPT (embeddings, blocks, cross entropy).
"""

from __future__ import annotations

import ctypes
import math

import torch

from limn_amd.seam import Node, Op, Tensor, active_device, bfloat16, capture, float16, float32, grad, int32, nn, optim, realize, set_device

TYPES = {"f32": float32, "f16": float16, "bf16": bfloat16}
TORCH = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
OF_LIMN = {float32: torch.float32, float16: torch.float16, bfloat16: torch.bfloat16, int32: torch.int32}
TYPESTR = {torch.float32: "<f4", torch.float16: "<f2", torch.bfloat16: "<i2", torch.int32: "<i4"}
GPT_VOCAB = 256


def listed():
    return [
        # the attention of one layer of the GPT training step (bench.py's C5): many short heads
        dict(name="attn_bf16_short", kind="attention", dtype="bf16", batch=32, heads=8, t_q=512, t_k=512, dim=64, causal=True, masked=False, train=True),
        # long-context training attention (bench.py's headline, C4)
        dict(name="attn_bf16_long", kind="attention", dtype="bf16", batch=8, heads=16, t_q=4096, t_k=4096, dim=128, causal=True, masked=False, train=True),
        # limn's own attention benchmark: 8192 tokens, 6 heads of 32, limn's default type
        dict(name="attn_f32", kind="attention", dtype="f32", batch=8, heads=6, t_q=1024, t_k=1024, dim=32, causal=True, masked=False, train=True),
        # the smallest attention step: a small float32 model (bench.py's C1)
        dict(name="attn_f32_small", kind="attention", dtype="f32", batch=2, heads=4, t_q=256, t_k=256, dim=64, causal=True, masked=False, train=True),
        # serving an encoder-decoder: a few hundred queries over padded keys, head dim 80, ragged lengths
        dict(name="attn_f16_cross", kind="attention", dtype="f16", batch=16, heads=16, t_q=197, t_k=1021, dim=80, causal=False, masked=True, train=False),
        # a feed-forward block in limn's default type
        dict(name="mlp_f32", kind="mlp", dtype="f32", batch=1, rows=4096, width=512, hidden=2048, out=512, act="relu"),
        # the smallest training step: a digit classifier on a small batch
        dict(name="mlp_f32_small", kind="mlp", dtype="f32", batch=1, rows=64, width=784, hidden=128, out=10, act="relu"),
        # the feed-forward block of the GPT training step
        dict(name="mlp_bf16", kind="mlp", dtype="bf16", batch=32, rows=512, width=512, hidden=2048, out=512, act="gelu"),
        # a large dense product (bench.py's C3)
        dict(name="matmul_bf16", kind="matmul", dtype="bf16", m=4096, k=4096, n=4096),
        # softmax then LayerNorm over long rows (bench.py's C2)
        dict(name="softmax_norm", kind="norm", rows=8192, width=8192),
        # one optimizer step
        dict(name="adamw", kind="adamw", width=1024),
        # the whole model, forward and backward, at the widths of the GPT training step
        dict(name="gpt_bf16", kind="gpt", dtype="bf16", layers=2, batch=32, ctx=512, width=512, heads=8),
    ]


def _span(rng, lo, hi, odd=0.4):
    """A size between lo and hi, even over its logarithm; a multiple of 16 but for `odd` of the draws."""
    x = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    return x if rng.random() < odd else min(hi, max(16, x // 16 * 16))


def draw(rng):
    kind = rng.choice(["attention", "attention", "attention", "matmul", "matmul", "mlp", "mlp", "norm", "adamw", "gpt"])
    if kind == "attention":
        dtype = rng.choice(["bf16", "f16", "f32", "f32"])
        causal, train = rng.random() < 0.6, rng.random() < 0.6
        t_q = _span(rng, 32, 4096 if dtype != "f32" else 2048)
        t_k = t_q if causal else _span(rng, 32, 4096 if dtype != "f32" else 2048)
        dim = rng.choice([16, 32, 64, 64, 80, 96, 128, 128])
        most = (1 << 35) if dtype != "f32" else (1 << 31)  # multiplications of one product over all heads
        pairs = max(1, min(256, most // (t_q * t_k * dim)))
        heads = rng.choice([h for h in (1, 2, 3, 4, 6, 8, 12, 16) if h <= pairs])
        batch = max(1, int(round(math.exp(rng.uniform(0, math.log(max(1, min(32, pairs // heads))))))))
        return dict(kind=kind, dtype=dtype, batch=batch, heads=heads, t_q=t_q, t_k=t_k, dim=dim, causal=causal, masked=rng.random() < 0.3, train=train)
    if kind == "matmul":
        dtype = rng.choice(["bf16", "bf16", "f16", "f32", "f32"])
        m, k, n = (_span(rng, 33, 2048 if dtype == "f32" else 4096) for _ in range(3))
        while m * k * n > 1 << 33:
            m, k, n = max(33, m // 2), k, max(33, n // 2)
        return dict(kind=kind, dtype=dtype, m=m, k=k, n=n)
    if kind == "mlp":
        dtype = rng.choice(["f32", "f32", "bf16"])
        batch = rng.choice([1, 1, 4, 16])
        rows = max(1, _span(rng, 32, 4096) // batch) if dtype == "f32" else max(16, _span(rng, 64, 16384) // batch)
        width, hidden = _span(rng, 32, 1024, 0.25), _span(rng, 32, 2048, 0.25)
        out = rng.choice([10, width, width, _span(rng, 16, 512)])
        return dict(kind=kind, dtype=dtype, batch=batch, rows=rows, width=width, hidden=hidden, out=out, act=rng.choice(["relu", "gelu"]))
    if kind == "norm":
        return dict(kind=kind, rows=_span(rng, 32, 8192), width=_span(rng, 64, 8192))
    if kind == "adamw":
        return dict(kind=kind, width=_span(rng, 32, 1024))
    heads = rng.choice([2, 4, 8])
    return dict(kind="gpt", dtype=rng.choice(["bf16", "bf16", "f32"]), layers=rng.choice([1, 2]), batch=rng.choice([1, 2, 3, 4, 8]),
                ctx=_span(rng, 33, 256), width=heads * rng.choice([16, 32, 64]), heads=heads)


# ---- inputs, the same for the framework and for the float64 reference -----------------------------


def _inputs(case, seed):
    """Name -> torch tensor on the GPU, from the seed alone, in the order a pass takes them."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)

    def normal(*shape, std=1.0, dtype=torch.float32):
        return (torch.randn(shape, generator=g, device="cuda") * std).to(dtype)

    def uniform(out, *fan):
        """A Linear's weight or bias as nn.Linear draws it."""
        bound = fan[-1] ** -0.5
        return (torch.rand((out, *fan[:-1]), generator=g, device="cuda") * 2 - 1) * bound

    kind = case["kind"]
    if kind == "attention":
        t = TORCH[case["dtype"]]
        lead = (case["batch"], case["heads"])
        got = dict(q=normal(*lead, case["t_q"], case["dim"], dtype=t), k=normal(*lead, case["t_k"], case["dim"], dtype=t),
                   v=normal(*lead, case["t_k"], case["dim"], dtype=t))
        if case["masked"]:  # keys padded to the longest of the batch: a tail of hidden ones, never all
            live = torch.randint((case["t_k"] + 1) // 2, case["t_k"] + 1, (case["batch"], 1, 1), generator=g, device="cuda")
            got["mask"] = (torch.arange(case["t_k"], device="cuda") < live).expand(*lead, case["t_k"]).to(t).contiguous()
        if case["train"]:
            got["dout"] = normal(*lead, case["t_q"], case["dim"], dtype=t)
        return got
    if kind == "matmul":
        t = TORCH[case["dtype"]]
        return dict(a=normal(case["m"], case["k"], std=0.125, dtype=t), b=normal(case["k"], case["n"], std=0.125, dtype=t))
    if kind == "mlp":
        t = TORCH[case["dtype"]]
        lead = (case["rows"],) if case["batch"] == 1 else (case["batch"], case["rows"])
        return dict(x=normal(*lead, case["width"], dtype=t), up=uniform(case["hidden"], case["width"], case["width"]), up_bias=uniform(case["hidden"], case["width"]),
                    down=uniform(case["out"], case["hidden"], case["hidden"]), down_bias=uniform(case["out"], case["hidden"]), dy=normal(*lead, case["out"], dtype=t))
    if kind == "norm":
        return dict(x=normal(case["rows"], case["width"]), weight=1 + normal(case["width"], std=0.1), bias=normal(case["width"], std=0.1))
    if kind == "adamw":
        d, got = case["width"], {}
        for name, shape in (("norm", (d,)), ("norm_bias", (d,)), ("qkv", (3 * d, d)), ("qkv_bias", (3 * d,)), ("proj", (d, d)), ("proj_bias", (d,)),
                            ("up", (4 * d, d)), ("up_bias", (4 * d,)), ("down", (d, 4 * d)), ("down_bias", (d,))):
            got[name] = normal(*shape, std=0.02)
            got["d_" + name] = normal(*shape, std=0.001)
        return got
    d, got = case["width"], dict()
    stream = torch.randint(0, GPT_VOCAB, (case["batch"], case["ctx"] + 1), generator=g, device="cuda", dtype=torch.int32)
    got["tokens"], got["targets"] = stream[:, :-1].contiguous(), stream[:, 1:].contiguous()
    got["tok.weight"], got["pos.weight"] = normal(GPT_VOCAB, d), normal(case["ctx"], d)
    for i in range(case["layers"]):
        for ln in ("ln1", "ln2"):
            got[f"{i}.{ln}.weight"], got[f"{i}.{ln}.bias"] = 1 + normal(d, std=0.1), normal(d, std=0.1)
        for name, o, n in (("qkv", 3 * d, d), ("proj", d, d), ("up", 4 * d, d), ("down", d, 4 * d)):
            got[f"{i}.{name}.weight"], got[f"{i}.{name}.bias"] = uniform(o, n, n), uniform(o, n)
    got["ln.weight"], got["ln.bias"], got["head.weight"] = 1 + normal(d, std=0.1), normal(d, std=0.1), uniform(GPT_VOCAB, d, d)
    return got


# ---- between torch's memory and limn's buffers -----------------------------------------------------


class _Bytes:
    """A limn device buffer as torch takes foreign memory; torch keeps this object, and so the buffer, alive."""

    __slots__ = ("buffer", "__cuda_array_interface__")

    def __init__(self, buffer, dtype, shape):
        self.buffer = buffer
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": TYPESTR[dtype], "data": (buffer.ptr, False), "version": 2}


def _as_torch(tensor):
    """A realized limn tensor's buffer as a torch tensor (no copy)."""
    dtype = OF_LIMN[tensor.dtype]
    got = torch.as_tensor(_Bytes(tensor.node.arg, dtype, tensor.shape), device="cuda")
    return got.view(torch.bfloat16) if dtype is torch.bfloat16 else got


def _as_limn(x, requires_grad=False):
    """A limn tensor in a device buffer of its own, holding x's values."""
    dtype = next(l for l, t in OF_LIMN.items() if t is x.dtype)
    buffer = active_device().alloc(x.numel() * x.element_size())
    t = Tensor.from_node(Node(Op.BUFFER, (), dtype, tuple(x.shape), buffer))
    t.requires_grad = requires_grad
    _as_torch(t).copy_(x)
    return t


# ---- what a program of each kind does in a pass ----------------------------------------------------


def _step(case):
    """The function such a program captures: limn tensors in, realized limn tensors out."""
    kind = case["kind"]
    if kind == "attention":
        causal, masked = case["causal"], case["masked"]

        def attention(q, k, v, *rest):
            out = q.attention(k, v, causal=causal, key_mask=rest[0] if masked else None)
            got = [out, *grad((out * rest[-1]).sum(), [q, k, v])]
            realize(*got)
            return got

        return attention
    if kind == "matmul":

        def matmul(a, b):
            return (a @ b).relu().realize()

        return matmul
    if kind == "mlp":
        from limn_amd.gpt import gelu, mixed

        up, down = nn.Linear(case["width"], case["hidden"]), nn.Linear(case["hidden"], case["out"])
        act = gelu if case["act"] == "gelu" else Tensor.relu

        def mlp(x, w1, b1, w2, b2, dy):
            up.weight, up.bias, down.weight, down.bias = w1, b1, w2, b2
            y = mixed(down, act(mixed(up, x)))
            got = [y, *grad((y * dy).sum(), [x, w1, b1, w2, b2])]
            realize(*got)
            return got

        return mlp
    if kind == "norm":
        norm = nn.LayerNorm(case["width"])

        def softmax_norm(x, weight, bias):
            norm.weight, norm.bias = weight, bias
            return norm(x.softmax(-1)).realize()

        return softmax_norm
    from limn_amd.gpt import GPT, GPTConfig, cross_entropy

    model = GPT(GPTConfig(vocab=GPT_VOCAB, ctx=case["ctx"], dim=case["width"], layers=case["layers"], heads=case["heads"], batch=case["batch"],
                          dtype=TYPES[case["dtype"]]))
    places = [(model.tok, "weight"), (model.pos, "weight")]
    for block in model.blocks:
        places += [(m, a) for m in (block.ln1, block.ln2, block.qkv, block.proj, block.up, block.down) for a in ("weight", "bias")]
    places += [(model.ln, "weight"), (model.ln, "bias"), (model.head, "weight")]

    def gpt(tokens, targets, *weights):
        for (module, attr), w in zip(places, weights):
            setattr(module, attr, w)
        logits = model(tokens)
        loss = cross_entropy(logits, targets)
        got = [logits, loss, *grad(loss, list(weights))]
        realize(*got)
        return got

    return gpt


_programs = {}  # configuration -> its captured step, as a program holds one for its whole run


def _program(case, args):
    key = tuple(sorted((k, v) for k, v in case.items() if k != "name"))
    if key not in _programs:
        _programs[key] = program = capture(_step(case))
        for _ in range(2):  # the two calls that capture observes
            program(*args)
    return _programs[key]


def _device():
    import limn_amd.hip  # noqa: F401  (registers "hip")

    try:
        return active_device()
    except RuntimeError:
        set_device("hip")
        return active_device()


def prepare(case, seed):
    device = _device()
    inputs = _inputs(case, seed)
    if case["kind"] == "attention" and not case["train"]:  # a server's call of the C ABI
        shape = (case["batch"], case["heads"], case["t_q"])
        out = torch.empty(*shape, case["dim"], device="cuda", dtype=TORCH[case["dtype"]])
        lse = torch.empty(*shape, device="cuda")
        return dict(entry=device.lib.limn_hip_sdpa_fwd, inputs=inputs, out=out, lse=lse, case=case)
    if case["kind"] == "adamw":
        names = [n for n in inputs if not n.startswith("d_")]
        params = [_as_limn(inputs[n], requires_grad=True) for n in names]
        grads = [_as_limn(inputs["d_" + n]) for n in names]
        opt = optim.AdamW(params, lr=3e-4, weight_decay=0.1)

        def update(*gs):
            opt.zero_grad()
            for p, g in zip(params, gs):
                p.grad = g
            opt.step()
            opt.zero_grad()
            return params

        program = capture(update)
        for _ in range(2):
            program(*grads)
        return dict(program=program, args=grads, outputs=[t for p in params for t in (p, *opt.moments[id(p)])])
    leaves = {"attention": "qkv", "mlp": ("x", "up", "up_bias", "down", "down_bias"), "gpt": [n for n in inputs if "." in n]}.get(case["kind"], ())
    args = [_as_limn(x, requires_grad=name in leaves) for name, x in inputs.items()]
    return dict(program=_program(case, args), args=args)


def run(state):
    if "entry" in state:
        c, x = state["case"], state["inputs"]
        mask = x["mask"].data_ptr() if c["masked"] else None
        status = state["entry"](x["q"].data_ptr(), x["k"].data_ptr(), x["v"].data_ptr(), mask, state["out"].data_ptr(), state["lse"].data_ptr(),
                                {"f32": 1, "f16": 2, "bf16": 3}[c["dtype"]], c["batch"] * c["heads"], c["t_q"], c["t_k"], c["dim"], c["dim"], int(c["causal"]),
                                c["dim"] ** -0.5, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
        if status != 0:
            raise RuntimeError(f"limn_hip_sdpa_fwd: status {status}")
        return [state["out"], state["lse"]]
    got = state["program"](*state["args"])
    if "outputs" in state:
        return [_as_torch(t) for t in state["outputs"]]
    return [_as_torch(t) for t in (got if isinstance(got, (list, tuple)) else [got])]


# ---- the work no implementation can do without -----------------------------------------------------


def work(case):
    kind, size = case["kind"], {"f32": 4, "f16": 2, "bf16": 2}.get(case.get("dtype"), 4)
    if kind == "attention":
        pairs = case["batch"] * case["heads"]
        unit = 2.0 * pairs * case["t_q"] * case["t_k"] * case["dim"] * (0.5 if case["causal"] else 1.0)
        q, k = pairs * case["t_q"] * case["dim"] * size, pairs * case["t_k"] * case["dim"] * size
        mask = pairs * case["t_k"] * size if case["masked"] else 0
        if case["train"]:  # q, k, v, dout in; out, dq, dk, dv out
            return dict(bytes=4 * q + 4 * k + mask, flops=7 * unit)
        return dict(bytes=2 * q + 2 * k + mask + pairs * case["t_q"] * 4, flops=2 * unit)
    if kind == "matmul":
        m, k, n = case["m"], case["k"], case["n"]
        return dict(bytes=(m * k + k * n + m * n) * size, flops=2.0 * m * k * n)
    if kind == "mlp":
        rows, weights = case["batch"] * case["rows"], case["hidden"] * (case["width"] + case["out"])
        # x and dy in, y and dx out; the float32 weights and their gradients
        return dict(bytes=2 * rows * (case["width"] + case["out"]) * size + 2 * weights * 4, flops=6.0 * rows * weights)
    if kind == "norm":
        return dict(bytes=2 * case["rows"] * case["width"] * 4, flops=10.0 * case["rows"] * case["width"])
    if kind == "adamw":  # p, m, v, g in; p, m, v out
        count = 12 * case["width"] ** 2 + 11 * case["width"]
        return dict(bytes=28 * count, flops=15.0 * count)
    d, tokens = case["width"], case["batch"] * case["ctx"]
    weights = case["layers"] * 12 * d * d + d * GPT_VOCAB
    flops = 6.0 * tokens * weights + case["layers"] * 7.0 * tokens * case["ctx"] * d
    return dict(bytes=2 * 4 * (weights + (GPT_VOCAB + case["ctx"]) * d) + tokens * GPT_VOCAB * size, flops=flops)


def tolerance(case):
    kind, dtype = case["kind"], case.get("dtype", "f32")
    if kind == "gpt":
        return {"rel": 2e-2, "max": 0.5} if dtype == "bf16" else {"rel": 1e-5, "max": 1e-3}
    if dtype == "bf16":
        return {"rel": 1e-2, "max": 0.2}
    if dtype == "f16":
        return {"rel": 2e-3, "max": 0.05}
    return {"rel": 1e-5, "max": 5e-4}


# ---- the same values in float64 --------------------------------------------------------------------


def _attend(q, k, v, causal, mask=None):
    """Attention over (..., t, d) in float64."""
    s = q @ k.transpose(-1, -2).contiguous() * q.shape[-1] ** -0.5
    if causal:
        s = s.masked_fill(torch.ones(s.shape[-2:], dtype=torch.bool, device=s.device).triu(1), -math.inf)
    if mask is not None:
        s = s.masked_fill((mask == 0).unsqueeze(-2), -math.inf)
    return torch.softmax(s, -1) @ v, torch.logsumexp(s.detach(), -1)


def _gelu(x):
    return 0.5 * x * (1 + torch.tanh(math.sqrt(2 / math.pi) * (x + 0.044715 * x**3)))


def exact(case, seed):
    kind, x = case["kind"], _inputs(case, seed)
    x = {n: t.double() if t.is_floating_point() else t for n, t in x.items()}
    if kind == "attention":
        parts = []
        for b in range(case["batch"]):
            for h in range(0, case["heads"], 4):  # a few heads at a time: the scores are large
                q, k, v = (x[n][b, h : h + 4].clone().requires_grad_(case["train"]) for n in "qkv")
                out, lse = _attend(q, k, v, case["causal"], x["mask"][b, h : h + 4] if case["masked"] else None)
                if case["train"]:
                    parts.append([out.detach(), *torch.autograd.grad(out, (q, k, v), x["dout"][b, h : h + 4])])
                else:
                    parts.append([out, lse])
        lead = (case["batch"], case["heads"])
        return [torch.cat(p).reshape(*lead, *p[0].shape[1:]) for p in zip(*parts)]
    if kind == "matmul":
        return [torch.relu(x["a"] @ x["b"])]
    if kind == "mlp":
        leaves = [x[n].requires_grad_() for n in ("x", "up", "up_bias", "down", "down_bias")]
        act = _gelu if case["act"] == "gelu" else torch.relu
        y = act(leaves[0] @ leaves[1].T + leaves[2]) @ leaves[3].T + leaves[4]
        return [y.detach(), *torch.autograd.grad(y, leaves, x["dy"])]
    if kind == "norm":
        y = torch.softmax(x["x"], -1)
        return [torch.nn.functional.layer_norm(y, y.shape[-1:], x["weight"], x["bias"], 1e-5)]
    if kind == "adamw":  # the two steps that capture observed, then the pass
        got = []
        for n in (n for n in x if not n.startswith("d_")):
            p, g = x[n], x["d_" + n]
            m, v = torch.zeros_like(p), torch.zeros_like(p)
            for step in (1, 2, 3):
                m, v = 0.9 * m + 0.1 * g, 0.999 * v + 0.001 * g * g
                p = p * (1 - 3e-4 * 0.1) - 3e-4 * (m / (1 - 0.9**step)) / (torch.sqrt(v / (1 - 0.999**step)) + 1e-8)
            got += [p, m, v]
        return got
    d, heads = case["width"], case["heads"]
    w = {n: t.requires_grad_() for n, t in x.items() if "." in n}
    h = w["tok.weight"][x["tokens"].long()] + w["pos.weight"]
    b, t = h.shape[:2]

    def norm(v, name):
        return torch.nn.functional.layer_norm(v, (d,), w[name + ".weight"], w[name + ".bias"], 1e-5)

    def linear(v, name):
        return v @ w[name + ".weight"].T + w[name + ".bias"]

    for i in range(case["layers"]):
        q, k, v = linear(norm(h, f"{i}.ln1"), f"{i}.qkv").reshape(b, t, 3, heads, d // heads).permute(2, 0, 3, 1, 4).contiguous()
        att = _attend(q, k, v, True)[0].transpose(1, 2).reshape(b, t, d)
        h = h + linear(att, f"{i}.proj")
        h = h + linear(_gelu(linear(norm(h, f"{i}.ln2"), f"{i}.up")), f"{i}.down")
    logits = norm(h, "ln") @ w["head.weight"].T
    loss = torch.nn.functional.cross_entropy(logits.reshape(-1, GPT_VOCAB), x["targets"].reshape(-1).long())
    return [logits.detach(), loss.detach(), *torch.autograd.grad(loss, list(w.values()))]
