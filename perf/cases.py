"""The work that a serving engine has this framework do, as timed cases.

Each case is one call into the layers that a model runner uses: a W8A8
linear, the gated MLP, an MoE block, the W8A8 part of a whole decoder layer
and the standalone quantizer.  ``listed`` names the fixed cases, ``draw``
gives more of the same ranges.  Decode batches (``graph``) are captured once
and replayed with fresh inputs copied into the static buffers, as the engine
runs them; prefill batches are eager calls.

Weights are int8 with a normal distribution (a row's largest magnitude about
127, as per-channel quantization leaves it) and scales that keep outputs near
unit size; activations are N(0, 1) in bf16 with 0.1% of the entries 20 times
larger.
"""

import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mini-sglang-fork_amd"))

from minisgl_amd.core import Context, set_global_ctx  # noqa: E402
from minisgl_amd.kernel import quant_per_token  # noqa: E402
from minisgl_amd.layers import (  # noqa: E402
    GatedMLPW8A8,
    LinearOProj,
    LinearQKVMerged,
    LinearReplicated,
    MoELayer,
    RMSNorm,
    RMSNormFused,
    RMSNormQuant,
)
from minisgl_amd.moe import create_moe_backend  # noqa: E402

DEV = "cuda:0"
HEAD = 128
EPS = 1e-6

# hidden, intermediate, query heads, key/value heads
QWEN3_0_6B = dict(hidden=1024, inter=3072, heads=16, kv=8)
QWEN3_14B = dict(hidden=5120, inter=17408, heads=40, kv=8)
QWEN3_32B = dict(hidden=5120, inter=25600, heads=64, kv=8)
QWEN3_32B_TP4 = dict(hidden=5120, inter=6400, heads=16, kv=2)  # one of four ranks' share
QWEN3_30B_A3B = dict(experts=128, topk=8, hidden=2048, inter=768)

# decode batches up to this size are captured in a graph by the engine
GRAPH_MAX = 256


def listed():
    return [
        # the smallest call: a decode batch through one projection of a small model, eagerly
        dict(name="linear_m16_small", kind="linear", m=16, k=1024, n=6144, bias=False, graph=False),
        # one token through a decoder layer's projections and norms: the latency of single-stream decode
        dict(name="layer_decode_m1", kind="layer", m=1, graph=True, **QWEN3_14B),
        # a full decode batch through the same layer
        dict(name="layer_decode_m64", kind="layer", m=64, graph=True, **QWEN3_14B),
        # the ragged tail of a chunked prefill through qkv with a bias
        dict(name="linear_m333_bias", kind="linear", m=333, k=5120, n=7168, bias=True, graph=False),
        # a short prompt through the MLP
        dict(name="mlp_m512", kind="mlp", m=512, act="silu", graph=False, hidden=5120, inter=17408),
        # an odd batch through a small model's MLP, with the other activation
        dict(name="mlp_m777_gelu", kind="mlp", m=777, act="gelu", graph=False, hidden=1024, inter=3072),
        # 32 decode tokens beside a 2048-token prefill chunk through a whole layer
        dict(name="layer_mixed_m2080", kind="layer", m=2080, graph=False, **QWEN3_32B),
        # the largest prefill batch through the MLP
        dict(name="mlp_m8192", kind="mlp", m=8192, act="silu", graph=False, hidden=5120, inter=17408),
        # mixture of experts: a decode batch, a ragged short prefill, a full prefill chunk
        dict(name="moe_decode_m16", kind="moe", m=16, graph=True, **QWEN3_30B_A3B),
        dict(name="moe_m300", kind="moe", m=300, graph=False, **QWEN3_30B_A3B),
        dict(name="moe_m4096", kind="moe", m=4096, graph=False, **QWEN3_30B_A3B),
        # the quantizer by itself on a large prefill's MLP activation
        dict(name="quant_8192x17408", kind="quant", m=8192, k=17408),
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choices(["linear", "mlp", "moe", "layer", "quant"], [5, 4, 4, 2, 1])[0]
    m = _log_int(rng, 1, 8192)
    graph = m <= GRAPH_MAX and kind in ("layer", "moe")
    if kind == "linear":
        sizes = []
        for c in (QWEN3_0_6B, QWEN3_14B, QWEN3_32B, QWEN3_32B_TP4):
            h, i, qkv = c["hidden"], c["inter"], (c["heads"] + 2 * c["kv"]) * HEAD
            sizes += [(h, qkv), (c["heads"] * HEAD, h), (h, 2 * i), (i, h)]
        if rng.random() < 0.5:
            k, n = rng.choice(sizes)
        else:
            step = rng.choice([16, 64, 128])
            k, n = step * _log_int(rng, 512 // step, 16384 // step), 8 * _log_int(rng, 64, 4096)
        while m * k * n > 8192 * 5120 * 17408:
            m = m // 2
        return dict(kind="linear", m=m, k=k, n=n, bias=rng.random() < 0.3, graph=m <= GRAPH_MAX and rng.random() < 0.5)
    if kind == "mlp":
        c = rng.choice([QWEN3_0_6B, QWEN3_14B, QWEN3_32B, QWEN3_32B_TP4])
        if c is QWEN3_32B:
            m = min(m, 5000)
        act = rng.choice(["silu", "silu", "gelu"])
        return dict(kind="mlp", m=m, act=act, graph=m <= GRAPH_MAX and rng.random() < 0.5, hidden=c["hidden"], inter=c["inter"])
    if kind == "moe":
        c = dict(QWEN3_30B_A3B)
        if rng.random() < 0.4:
            c = dict(experts=rng.choice([16, 32, 64, 128]), topk=rng.choice([2, 4, 6, 8]), hidden=rng.choice([1024, 2048, 4096]),
                     inter=16 * _log_int(rng, 16, 96))
        return dict(kind="moe", m=m, graph=graph, **c)
    if kind == "layer":
        c = rng.choice([QWEN3_0_6B, QWEN3_14B, QWEN3_32B, QWEN3_32B_TP4])
        return dict(kind="layer", m=min(m, 3500), graph=graph, **c)
    return dict(kind="quant", m=m, k=8 * _log_int(rng, 64, 3200))


# ------------------------------------------------------------------ inputs
def _acts(m, k, gen):
    x = torch.randn(m, k, generator=gen, device=DEV)
    x = torch.where(torch.rand(m, k, generator=gen, device=DEV) < 1e-3, x * 20, x)
    return x.to(torch.bfloat16)


def _weight(shape, gen):
    w = torch.empty(shape, dtype=torch.int8, device=DEV)
    flat = w.view(-1, shape[-1])
    step = max(1, (1 << 27) // shape[-1])
    for r in range(0, flat.shape[0], step):
        part = flat[r : r + step]
        part.copy_((torch.randn(part.shape, generator=gen, device=DEV) * 33).round_().clamp_(-127, 127))
    return w


def _scale(shape, k, gen):
    return (torch.rand(shape, generator=gen, device=DEV) + 0.5) / (33 * math.sqrt(k))


def _norm(layer, gen):
    size = layer.weight.shape[0]
    layer.load_state_dict({"weight": (torch.rand(size, generator=gen, device=DEV) + 0.5).to(torch.bfloat16)})
    return layer


def _linear(layer, gen):
    n, k = layer.weight.shape
    sd = {"weight": _weight((n, k), gen), "weight_scale": _scale((n,), k, gen)}
    if layer.bias is not None:
        sd["bias"] = torch.randn(n, generator=gen, device=DEV).to(torch.bfloat16)
    layer.load_state_dict(sd)
    return layer


def _mlp(hidden, inter, act, gen):
    mlp = GatedMLPW8A8(hidden, inter, hidden_act=act)
    _linear(mlp.gate_up_proj, gen)
    _linear(mlp.down_proj, gen)
    return mlp


class _DecoderLayer:
    """The W8A8 part of a Qwen3 decoder layer; the attention between qkv and
    o_proj is not this framework's, so o_proj takes the normed queries."""

    def __init__(self, c, gen):
        self.heads, self.kv = c["heads"], c["kv"]
        self.norm1 = _norm(RMSNormQuant(c["hidden"], EPS), gen)
        self.qkv = _linear(LinearQKVMerged(c["hidden"], HEAD, self.heads, self.kv, has_bias=False), gen)
        self.q_norm = _norm(RMSNorm(HEAD, EPS), gen)
        self.k_norm = _norm(RMSNorm(HEAD, EPS), gen)
        self.o = _linear(LinearOProj(self.heads * HEAD, c["hidden"], has_bias=False), gen)
        self.norm2 = _norm(RMSNormFused(c["hidden"], EPS), gen)
        self.mlp = _mlp(c["hidden"], c["inter"], "silu", gen)

    def forward(self, x):
        # x is the residual stream, which the second norm updates in place
        q8, s, residual = self.norm1.forward(x)
        qkv = self.qkv.forward_quantized(q8, s)
        q, k, v = qkv.split([self.heads * HEAD, self.kv * HEAD, self.kv * HEAD], dim=-1)
        self.q_norm.forward_inplace(q.view(-1, self.heads, HEAD))
        self.k_norm.forward_inplace(k.view(-1, self.kv, HEAD))
        h, residual = self.norm2.forward(self.o.forward(q), residual)
        return self.mlp.forward(h), residual, k, v


class _MoEBlock:
    """The norm before a mixture of experts and the experts."""

    def __init__(self, c, gen):
        e, h, i = c["experts"], c["hidden"], c["inter"]
        self.norm = _norm(RMSNorm(h, EPS), gen)
        self.moe = MoELayer(e, c["topk"], h, i)
        self.moe.load_state_dict({
            "gate_up_proj": _weight((e, 2 * i, h), gen), "down_proj": _weight((e, h, i), gen),
            "gate_up_scale": _scale((e, 2 * i), h, gen), "down_scale": _scale((e, h), i, gen),
        })

    def forward(self, x, logits):
        return self.moe.forward(self.norm.forward(x), logits)


def _inputs(case, gen):
    if case["kind"] in ("linear", "quant"):
        return (_acts(case["m"], case["k"], gen),)
    if case["kind"] == "moe":
        return _acts(case["m"], case["hidden"], gen), torch.randn(case["m"], case["experts"], generator=gen, device=DEV).to(torch.bfloat16)
    return (_acts(case["m"], case["hidden"], gen),)


def _model(case, gen):
    kind = case["kind"]
    if kind == "linear":
        return _linear(LinearReplicated(case["k"], case["n"], has_bias=case["bias"]), gen)
    if kind == "mlp":
        return _mlp(case["hidden"], case["inter"], case["act"], gen)
    if kind == "moe":
        return _MoEBlock(case, gen)
    return _DecoderLayer(case, gen)


def prepare(case, seed):
    gen = torch.Generator(device=DEV).manual_seed(seed)
    inputs = _inputs(case, gen)
    if case["kind"] == "quant":
        return {"call": quant_per_token, "inputs": inputs}
    set_global_ctx(Context(moe_backend=create_moe_backend("fused_w8a8")))
    model = _model(case, gen)
    if not case["graph"]:
        call = model.forward
        if case["kind"] == "layer":  # a fresh residual stream, as the layers before leave one
            call = lambda x: model.forward(x.clone())  # noqa: E731
        return {"call": call, "inputs": inputs}
    static = [t.clone() for t in inputs]
    model.forward(*static)  # an eager pass before the capture, as the engine does
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = model.forward(*static)
    return {"graph": graph, "static": static, "out": out, "inputs": inputs, "model": model}


def run(state):
    if "graph" not in state:
        return state["call"](*state["inputs"])
    for buf, x in zip(state["static"], state["inputs"]):
        buf.copy_(x)
    state["graph"].replay()
    return state["out"]


# ------------------------------------------------------------------ floors
def work(case):
    kind, m = case["kind"], case["m"]
    if kind == "quant":
        return {"bytes": m * (3 * case["k"] + 4), "flops": 3 * m * case["k"]}
    if kind == "linear":
        k, n = case["k"], case["n"]
        return {"bytes": 2 * m * k + n * k + 4 * n + 2 * m * n + (2 * n if case["bias"] else 0), "flops": 2 * m * n * k}
    h, i = case["hidden"], case["inter"]
    mlp_weights = 3 * h * i + 4 * (2 * i + h)
    if kind == "mlp":
        return {"bytes": 4 * m * h + mlp_weights, "flops": 6 * m * h * i}
    if kind == "moe":
        e, k = case["experts"], case["topk"]
        touched = e * (1 - (1 - k / e) ** m)
        return {"bytes": 4 * m * h + 2 * m * e + touched * mlp_weights, "flops": 6 * m * k * h * i}
    qn, kvn = case["heads"] * HEAD, case["kv"] * HEAD
    proj = h * (qn + 2 * kvn) + qn * h
    small = 4 * (qn + 2 * kvn + h) + 4 * h + 4 * HEAD
    return {"bytes": 6 * m * h + 4 * m * kvn + proj + small + mlp_weights, "flops": 2 * m * (proj + 3 * h * i)}


def tolerance(case):
    kind = case["kind"]
    if kind == "quant":
        return {"rel": 1e-6, "differ": 1e-6}
    if kind == "linear":
        return {"rel": 7e-3}
    return {"rel": 2.5e-2}


# ------------------------------------------------------- 64-bit references
def _quant64(x):
    s = x.abs().amax(dim=1, keepdim=True) / 127
    return torch.where(s > 0, (x / s).round(), 0.0).clamp(-127, 127), s


def _linear64(x, w, s_w, bias=None):
    q, s = _quant64(x)
    y = torch.empty(x.shape[0], w.shape[0], dtype=torch.float64, device=x.device)
    for r in range(0, w.shape[0], 8192):
        y[:, r : r + 8192] = q @ w[r : r + 8192].double().t()
    y = y * s * s_w.double()
    return y if bias is None else y + bias.double()


def _gated64(x, w1, s1, w2, s2, act):
    g, u = _linear64(x, w1, s1).chunk(2, dim=1)
    g = g * torch.sigmoid(g) if act == "silu" else 0.5 * g * (1 + torch.erf(g / math.sqrt(2)))
    return _linear64(g * u, w2, s2)


def _norm64(x, weight):
    return x * torch.rsqrt((x * x).mean(dim=-1, keepdim=True) + EPS) * weight.double()


def _mlp64(x, mlp, act):
    gu, dn = mlp.gate_up_proj, mlp.down_proj
    return _gated64(x, gu.weight, gu.weight_scale, dn.weight, dn.weight_scale, act)


def exact(case, seed):
    gen = torch.Generator(device=DEV).manual_seed(seed)
    inputs = _inputs(case, gen)
    x, kind = inputs[0].double(), case["kind"]
    if kind == "quant":
        q, s = _quant64(x)
        return q.to(torch.int8), s[:, 0]
    set_global_ctx(Context(moe_backend=create_moe_backend("fused_w8a8")))
    model = _model(case, gen)
    if kind == "linear":
        return _linear64(x, model.weight, model.weight_scale, model.bias)
    if kind == "mlp":
        return _mlp64(x, model, case["act"])
    if kind == "moe":
        h = _norm64(x, model.norm.weight)
        p, ids = torch.sort(torch.softmax(inputs[1].double(), dim=1), dim=1, descending=True, stable=True)
        p, ids = p[:, : case["topk"]], ids[:, : case["topk"]]
        p = p / p.sum(dim=1, keepdim=True)
        y, moe = torch.zeros_like(h), model.moe
        for e in range(case["experts"]):
            t, slot = (ids == e).nonzero(as_tuple=True)
            if t.numel():
                y.index_add_(0, t, p[t, slot, None] * _gated64(
                    h[t], moe.gate_up_proj[e], moe.gate_up_scale[e], moe.down_proj[e], moe.down_scale[e], "silu"))
        return y
    m, qn, kvn = case["m"], case["heads"] * HEAD, case["kv"] * HEAD
    qkv = _linear64(_norm64(x, model.norm1.weight), model.qkv.weight, model.qkv.weight_scale)
    q, k, v = qkv.split([qn, kvn, kvn], dim=1)
    q = _norm64(q.reshape(m, -1, HEAD), model.q_norm.weight).reshape(m, qn)
    k = _norm64(k.reshape(m, -1, HEAD), model.k_norm.weight).reshape(m, kvn)
    h = _linear64(q, model.o.weight, model.o.weight_scale) + x
    return _mlp64(_norm64(h, model.norm2.weight), model.mlp, "silu"), h, k, v
