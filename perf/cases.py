"""The work that this framework's speed is judged by: one pass of each operator family through its
public entry points, from single-token calls to the largest configurations, in every float type the
family is used in, on even and on ragged sizes.

A graph is planned once (`HipBackend.plan`), its inputs and weights are uploaded once and stay in
device memory, and a pass is one `HipPlan.launch()`, as in a serving or benchmark loop. The e4m3
linear is called on device pointers, and `plan_run` passes host data through `Plan.run`, the call
a frontend makes. Outputs stay in the plan's device buffers and are read with `HipPlan.output`.

Ranges (`draw`): softmax + argmax over 1 to 8192 rows of 1000 to 131072 columns; a fused map and sum
along either axis of up to 2^26 elements; products with 1 to 4096 rows, inner and outer sizes of 64
to 12288 and batches up to 16, in bf16, f16 and f32; attention over 1 to 4096 positions, 1 to 128
heads of 32, 64 or 128; e4m3 linears and 2/4/8-bit weight products of 1 to 2048 rows; gated MLPs of
1 to 2048 tokens; host-to-host f32 MLPs of 1 to 256 rows.
"""
import math
import types

import torch

import kurumi_amd as ku
from kurumi_amd import DType, Graph, Tensor

TYPES = {"f32": (DType.F32, torch.float32), "bf16": (DType.BF16, torch.bfloat16), "f16": (DType.F16, torch.float16),
         "i32": (DType.I32, torch.int32), "u8": (DType.U8, torch.uint8)}
TORCH_OF = {d: t for d, t in TYPES.values()}
_backend = None


def listed():
    return [
        # the row softmax and first-index argmax over a whole batch of vocabulary logits (the benchmark's headline)
        {"name": "softmax_8192x32000", "op": "softmax", "rows": 8192, "cols": 32000, "dtype": "f32"},
        # one decode step's logits: few rows, an odd vocabulary
        {"name": "softmax_4x50257", "op": "softmax", "rows": 4, "cols": 50257, "dtype": "f32"},
        # the fused map and sum of the benchmark, along the first axis: per-feature statistics of a batch
        {"name": "reduce_cols_16384x1000", "op": "reduce", "rows": 16384, "cols": 1000, "axis": 0, "dtype": "f32"},
        # an MLP projection over a prompt (the benchmark's bf16 product)
        {"name": "gemm_4096_bf16", "op": "gemm", "batch": 1, "m": 4096, "n": 11008, "k": 4096, "nt": False, "dtype": "bf16"},
        # the same projection for a batch of decoded tokens: bound by reading the weight
        {"name": "gemm_decode16_bf16", "op": "gemm", "batch": 1, "m": 16, "n": 11008, "k": 4096, "nt": False, "dtype": "bf16"},
        # the default element type, sizes that are no multiple of anything
        {"name": "gemm_ragged_f32", "op": "gemm", "batch": 1, "m": 1500, "n": 2001, "k": 1111, "nt": False, "dtype": "f32"},
        # causal self-attention over a prompt (the benchmark's attention)
        {"name": "attn_2048_bf16", "op": "attention", "b": 4, "h": 32, "s": 2048, "d": 128, "causal": True, "dtype": "bf16"},
        # an encoder's attention in the default element type, an odd length
        {"name": "attn_500_f32", "op": "attention", "b": 2, "h": 8, "s": 500, "d": 64, "causal": False, "dtype": "f32"},
        # the e4m3 linear layer over a prompt (the benchmark's), quantising its activation
        {"name": "linear_e4m3_2048", "op": "e4m3", "m": 2048, "n": 11008, "k": 4096, "dtype": "bf16"},
        # int4 weight-only projection of one decoded token
        {"name": "quant_int4_1", "op": "quant", "m": 1, "n": 11008, "k": 4096, "bits": 4, "group": 128, "sym": True, "dtype": "bf16"},
        # a norm and gated MLP of a block over a short prompt
        {"name": "mlp_300_bf16", "op": "mlp", "tokens": 300, "hidden": 2048, "inter": 5504, "dtype": "bf16"},
        # a small f32 classifier called on host data, as a frontend does: latency
        {"name": "plan_run_32", "op": "plan_run", "rows": 32, "d_in": 784, "hidden": 512, "d_out": 10, "dtype": "f32"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng, lo, hi, step=64):
    """A size spread over its logarithm: three in four a multiple of `step`, the others as they come."""
    v = _log(rng, lo, hi)
    return max(lo, v // step * step) if rng.random() < 0.75 else v


def _one(rng):
    op = rng.choice(["softmax", "reduce", "gemm", "gemm", "gemm", "attention", "attention", "e4m3", "quant", "quant", "mlp", "plan_run"])
    float_type = rng.choice(["bf16", "f16", "f32"])
    if op == "softmax":
        return {"op": op, "rows": _log(rng, 1, 8192), "cols": _size(rng, 1000, 131072), "dtype": rng.choice(["f32", "bf16"])}
    if op == "reduce":
        return {"op": op, "rows": _log(rng, 16, 65536), "cols": _size(rng, 16, 65536), "axis": rng.randrange(2), "dtype": rng.choice(["f32", "bf16"])}
    if op == "gemm":
        return {"op": op, "batch": rng.choice([1, 1, 1, _log(rng, 2, 16)]), "m": _log(rng, 1, 4096), "n": _size(rng, 64, 12288),
                "k": _size(rng, 64, 12288), "nt": rng.random() < 0.5, "dtype": float_type}
    if op == "attention":
        return {"op": op, "b": _log(rng, 1, 4), "h": _log(rng, 1, 32), "s": _log(rng, 1, 4096), "d": rng.choice([32, 64, 128]),
                "causal": rng.random() < 0.5, "dtype": float_type}
    if op == "e4m3":
        return {"op": op, "m": _log(rng, 1, 2048), "n": _size(rng, 64, 12288), "k": 128 * _log(rng, 1, 64), "dtype": float_type}
    if op == "quant":
        group = rng.choice([32, 64, 128])
        return {"op": op, "m": _log(rng, 1, 2048), "n": _size(rng, 64, 12288), "k": group * _log(rng, 4, 8192 // group),
                "bits": rng.choice([2, 4, 4, 8]), "group": group, "sym": rng.random() < 0.5, "dtype": float_type}
    if op == "mlp":
        return {"op": op, "tokens": _log(rng, 1, 2048), "hidden": _size(rng, 256, 4096), "inter": _size(rng, 512, 11008),
                "dtype": rng.choice(["bf16", "f16"])}
    return {"op": op, "rows": _log(rng, 1, 256), "d_in": _log(rng, 16, 2048), "hidden": _log(rng, 16, 2048), "d_out": _log(rng, 2, 1000),
            "dtype": "f32"}


def draw(rng):
    """No larger than the largest listed cases; in f32, whose matrix rate is a sixteenth, no more than 4e10 operations."""
    while True:
        c = _one(rng)
        w = work(c)
        if 2e4 < w["bytes"] <= 2.1e9 and w["flops"] <= (4e10 if c["dtype"] == "f32" else 3.7e11):
            return c


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) * 7919 + 17)


def _randn(gen, shape, std, dtype):
    return torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32).mul_(std).to(TYPES[dtype][1])


def _pack(q, bits):
    """Whole numbers [n, k] packed along k, low field first."""
    per = 8 // bits
    q = (q & ((1 << bits) - 1)).reshape(q.shape[0], -1, per)
    return sum(q[..., i] << (bits * i) for i in range(per)).to(torch.uint8)


def _inputs(case, seed):
    """The inputs as tensors on the GPU, made from the seed alone."""
    gen, c, dt = _generator(seed), types.SimpleNamespace(**case), case["dtype"]
    if c.op == "softmax":
        return {"x": _randn(gen, (c.rows, c.cols), 3.0, dt)}
    if c.op == "reduce":
        return {"x": _randn(gen, (c.rows, c.cols), 1.0, dt), "b": _randn(gen, (c.cols,), 0.5, dt)}
    if c.op == "gemm":
        lead = (c.batch,) if c.batch > 1 else ()
        return {"a": _randn(gen, lead + (c.m, c.k), 1.0, dt),
                "b": _randn(gen, lead + ((c.n, c.k) if c.nt else (c.k, c.n)), c.k ** -0.5, dt)}
    if c.op == "attention":
        return {n: _randn(gen, (c.b, c.h, c.s, c.d), 1.0, dt) for n in "qkv"}
    if c.op == "e4m3":
        w = _randn(gen, (c.n, c.k), 0.02, "f32")
        sw = w.abs().amax(1) / 448.0
        return {"x": _randn(gen, (c.m, c.k), 1.0, dt), "wq": (w / sw[:, None]).clamp_(-448, 448).to(torch.float8_e4m3fn), "sw": sw}
    if c.op == "quant":
        x = _randn(gen, (c.m, c.k), 1.0, dt)
        w = _randn(gen, (c.n, c.k // c.group, c.group), 0.02, "f32")
        top = (1 << (c.bits - 1)) - 1 if c.sym else (1 << c.bits) - 1
        low = torch.zeros_like(w[..., 0]) if c.sym else w.amin(2).half().float()
        scale = ((w.abs().amax(2) if c.sym else w.amax(2) - low) / top).half()
        q = ((w - low[..., None]) / scale.float()[..., None]).round_().clamp_(-top - 1 if c.sym else 0, top).to(torch.int32)
        got = {"x": x, "qw": _pack(q.reshape(c.n, c.k), c.bits), "scales": scale}
        return got if c.sym else dict(got, mins=low.half())
    if c.op == "mlp":
        return {"x": _randn(gen, (c.tokens, c.hidden), 1.0, dt), "gain": (1 + _randn(gen, (c.hidden,), 0.1, "f32")).to(TYPES[dt][1]),
                "gate": _randn(gen, (c.hidden, c.inter), c.hidden ** -0.5, dt), "up": _randn(gen, (c.hidden, c.inter), c.hidden ** -0.5, dt),
                "down": _randn(gen, (c.inter, c.hidden), c.inter ** -0.5, dt)}
    return {"x": _randn(gen, (c.rows, c.d_in), 1.0, dt), "w1": _randn(gen, (c.d_in, c.hidden), c.d_in ** -0.5, dt),
            "b1": _randn(gen, (c.hidden,), 0.1, dt), "w2": _randn(gen, (c.hidden, c.d_out), c.hidden ** -0.5, dt)}


def _bytes(t):
    return t.contiguous().reshape(-1).view(torch.uint8).cpu().numpy()


def _host(t, dtype):
    return Tensor(dtype, t.shape, _bytes(t))


def _read(t):
    """A host tensor of the library as a torch tensor."""
    return torch.frombuffer(bytearray(t.data), dtype=TORCH_OF[t.dtype]).reshape(t.shape)


class PlanOutputs(list):
    """A plan's outputs: they stay in the plan's own device buffers and are downloaded as they are read."""

    def __init__(self, plan, count):
        super().__init__(range(count))
        self.plan = plan

    def __getitem__(self, i):
        return _read(self.plan.output(i))

    def __iter__(self):
        return (self[i] for i in range(len(self)))


def _like(g, x, v):
    return g.broadcast_to(v, g.shape(x))


def _graph(case, seed):
    """(graph, {input node: host tensor}, roots)."""
    c, dt = types.SimpleNamespace(**case), TYPES[case["dtype"]][0]
    t, g, feeds = _inputs(case, seed), Graph(), {}

    def feed(name):
        n = g.input(list(t[name].shape), dt)
        feeds[n] = _host(t[name], dt)
        return n

    def const(name, dtype):
        return g.constant_bytes(dtype, _bytes(t[name]), list(t[name].shape))

    if c.op == "softmax":
        y = g.softmax(feed("x"), 1)
        roots = [y, g.cast(g.argmax(y, 1), DType.I32)]
    elif c.op == "reduce":
        x = feed("x")
        roots = [g.sum(g.mul(g.relu(g.add(g.mul(x, x), _like(g, x, feed("b")))), g.scalar(x, 0.5)), c.axis)]
    elif c.op == "gemm":
        a, b, r = feed("a"), feed("b"), 1 if c.batch > 1 else 0
        lead = [0] if r else []
        roots = [g.dot_general(a, b, [r + 1], [r + 1 if c.nt else r], lead, lead)]
    elif c.op == "attention":
        roots = [g.sdpa(feed("q"), feed("k"), feed("v"), c.causal)]
    elif c.op == "quant":
        mins = None if c.sym else const("mins", DType.F16)
        roots = [g.quant_matmul(feed("x"), const("qw", DType.U8), const("scales", DType.F16), mins, c.bits, c.group)]
    elif c.op == "mlp":
        x = feed("x")
        h = g.mul(g.rmsnorm(x, 1, 1e-6), _like(g, x, feed("gain")))
        roots = [g.matmul(g.mul(g.silu(g.matmul(h, feed("gate"))), g.matmul(h, feed("up"))), feed("down"))]
    else:
        x = feed("x")
        h = g.matmul(x, const("w1", dt))
        h = g.relu(g.add(h, _like(g, h, const("b1", dt))))
        roots = [g.softmax(g.matmul(h, const("w2", dt)), 1)]
    return g, feeds, roots


def prepare(case, seed):
    global _backend
    if _backend is None:  # one backend for the program
        _backend = ku.HipBackend()
    c = types.SimpleNamespace(**case)
    if c.op == "e4m3":
        t = _inputs(case, seed)
        y = torch.empty((c.m, c.n), dtype=TYPES[c.dtype][1], device="cuda")
        return types.SimpleNamespace(op=c.op, t=t, y=y, dt=TYPES[c.dtype][0], m=c.m, n=c.n, k=c.k)
    g, feeds, roots = _graph(case, seed)
    if c.op == "plan_run":
        return types.SimpleNamespace(op=c.op, g=g, feeds=feeds, plan=_backend.compile(g, roots[0]))
    plan = _backend.plan(g, roots, feeds)
    return types.SimpleNamespace(op=c.op, plan=plan, outputs=PlanOutputs(plan, len(roots)))


def run(state):
    s = state
    if s.op == "e4m3":
        _backend.linear_e4m3(s.t["x"].data_ptr(), s.dt, s.t["wq"].data_ptr(), s.t["sw"].data_ptr(), s.y.data_ptr(), s.dt, s.m, s.n, s.k)
        return s.y
    if s.op == "plan_run":
        return _read(s.plan.run(s.g, s.feeds))
    s.plan.launch()
    return s.outputs


def work(case):
    """Each input and weight read once, each output written once."""
    c = types.SimpleNamespace(**case)
    w = {"f32": 4}.get(c.dtype, 2)
    if c.op == "softmax":
        return {"bytes": c.rows * (2 * c.cols * w + 4), "flops": 0}
    if c.op == "reduce":
        return {"bytes": w * (c.rows * c.cols + c.cols + (c.rows if c.axis else c.cols)), "flops": 0}
    if c.op == "gemm":
        return {"bytes": w * c.batch * (c.m * c.k + c.k * c.n + c.m * c.n), "flops": 2 * c.batch * c.m * c.n * c.k}
    if c.op == "attention":
        return {"bytes": 4 * w * c.b * c.h * c.s * c.d, "flops": 4 * c.b * c.h * c.s * c.s * c.d // (2 if c.causal else 1)}
    if c.op == "e4m3":
        return {"bytes": c.m * c.k * w + c.n * c.k + 4 * c.n + c.m * c.n * w, "flops": 2 * c.m * c.n * c.k}
    if c.op == "quant":
        tables = (1 if c.sym else 2) * 2 * c.n * (c.k // c.group)
        return {"bytes": w * c.m * (c.k + c.n) + c.n * c.k * c.bits // 8 + tables, "flops": 2 * c.m * c.n * c.k}
    if c.op == "mlp":
        return {"bytes": w * (2 * c.tokens * c.hidden + c.hidden + 3 * c.hidden * c.inter), "flops": 6 * c.tokens * c.hidden * c.inter}
    return {"bytes": w * (c.rows * (c.d_in + c.d_out) + c.hidden * (c.d_in + c.d_out + 1)),
            "flops": 2 * c.rows * c.hidden * (c.d_in + c.d_out)}


def tolerance(case):
    """About four times the distance to the 64-bit result that was measured (the type's rounding of
    the result; sums in 32 bits). An argmax over a 16-bit softmax is compared as it is stored: the
    map before it does not depend on the order of a sum but through the last rounding."""
    op, dt = case["op"], case["dtype"]
    if op == "softmax":
        return {"rel": 4e-6 if dt == "f32" else 8e-3, "differ": 0.0 if dt == "f32" else 0.01}
    if dt != "bf16":
        return {"rel": (8e-3 if op == "mlp" else 2e-3) if dt == "f16" else 1e-5}
    return {"rel": 3e-2 if op == "mlp" else 1e-2}


def exact(case, seed):
    """What `run` returns, in 64 bits and without rounding between the steps."""
    c, t = types.SimpleNamespace(**case), {k: v for k, v in _inputs(case, seed).items()}
    if c.op == "e4m3":  # the quantised activation is part of what is asked for: by its definition, in 32 bits
        sx = t["x"].float().abs().amax() * (1.0 / 448.0)
        xq = (t["x"].float() * (1.0 / sx)).clamp_(-448, 448).to(torch.float8_e4m3fn)
        return (xq.double() @ t["wq"].double().t().contiguous()) * (sx.double() * t["sw"].double())
    d = {k: v.double() for k, v in t.items() if k != "qw"}
    if c.op == "softmax":
        return [torch.softmax(d["x"], 1), None]
    if c.op == "reduce":
        return [(torch.relu(d["x"] * d["x"] + d["b"]) * 0.5).sum(c.axis)]
    if c.op == "gemm":
        return [torch.matmul(d["a"], d["b"].transpose(-1, -2).contiguous() if c.nt else d["b"])]
    if c.op == "attention":
        out = torch.empty_like(d["q"])
        mask = torch.ones((c.s, c.s), dtype=torch.bool, device="cuda").triu(1) if c.causal else None
        for i in range(c.b):
            for j in range(c.h):
                p = (d["q"][i, j] @ d["k"][i, j].t().contiguous()) * (c.d ** -0.5)
                p = p if mask is None else p.masked_fill(mask, float("-inf"))
                out[i, j] = torch.softmax(p, 1) @ d["v"][i, j]
        return [out]
    if c.op == "quant":
        per, f = 8 // c.bits, t["qw"].int()[..., None] >> (torch.arange(8 // c.bits, device="cuda") * c.bits)
        q = (f & ((1 << c.bits) - 1)).reshape(c.n, -1, c.group)
        q = torch.where(q >= 1 << (c.bits - 1), q - (1 << c.bits), q) if c.sym else q
        w = q.double() * d["scales"][..., None] + (0.0 if c.sym else d["mins"][..., None])
        assert per * t["qw"].shape[1] == c.k
        return [d["x"] @ w.reshape(c.n, c.k).t().contiguous()]
    if c.op == "mlp":
        h = d["x"] * torch.rsqrt((d["x"] * d["x"]).mean(1, keepdim=True) + 1e-6) * d["gain"]
        return [(torch.nn.functional.silu(h @ d["gate"]) * (h @ d["up"])) @ d["down"]]
    return torch.softmax(torch.relu(d["x"] @ d["w1"] + d["b1"]) @ d["w2"], 1)
