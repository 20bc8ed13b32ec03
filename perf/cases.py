"""The work that a user of this framework has it do, as measurable cases.

LoRA training of an MQA decoder over frozen NF4 weights: single projections from a few rows to
a long packed batch, the q/k/v group with its rotary step, the MLP, a whole decoder layer, the
projection loss, the optimizer step, and the weight's encode (load time) and decode (export).
Every case calls the public entry points; `exact` restates the same arithmetic in 64 bits with
torch alone, from the inputs of `prepare`.
"""

import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "causal-tuner_amd"))

from causal_tuner.kernels.linear import project_group, projection_budget  # noqa: E402
from causal_tuner.kernels.loss import projection_loss  # noqa: E402
from causal_tuner.kernels.nf4_cuda import dequantize_nf4  # noqa: E402
from causal_tuner.modeling.decoder import DecoderConfig, Layer, record_positions, rotary_values  # noqa: E402
from causal_tuner.modeling.lora import Projection  # noqa: E402
from causal_tuner.modeling.mlp import MLP  # noqa: E402
from causal_tuner.optim import FusedAdamW  # noqa: E402
from causal_tuner.quant.nf4 import quantize_nf4  # noqa: E402

DEVICE = "cuda"
DTYPES = {"bf16": torch.bfloat16, "f32": torch.float32, "f16": torch.float16}
BUDGET = 1 << 30  # the projection budget (kept xa) that a training step gives each group
NF4_BYTES = 0.5 + 1 / 64 + 1 / 4096  # packed codes and scales per weight element


def listed():
    return [
        # One small adapter on a short sequence (512 tokens, rank 16): launches and host path.
        {"name": "projection-small", "kind": "projection", "rows": 512, "inputs": 1024, "outputs": 1024,
         "rank": 16, "bias": False, "keep": False, "dtype": "bf16"},
        # A wide projection over a handful of tokens: the packed weight's stream is the work.
        {"name": "projection-few-rows", "kind": "projection", "rows": 16, "inputs": 6144, "outputs": 24576,
         "rank": 256, "bias": False, "keep": True, "dtype": "bf16"},
        # A short, ragged prompt through the same kind of layer, the other way round.
        {"name": "projection-mid-rows", "kind": "projection", "rows": 251, "inputs": 24576, "outputs": 6144,
         "rank": 256, "bias": False, "keep": True, "dtype": "bf16"},
        # A long packed batch through the widest projection: the largest matrix products.
        {"name": "projection-long", "kind": "projection", "rows": 16384, "inputs": 6144, "outputs": 24576,
         "rank": 256, "bias": False, "keep": True, "dtype": "bf16"},
        # The float32 compute dtype (a model trained with --dtype float32).
        {"name": "projection-float32", "kind": "projection", "rows": 1000, "inputs": 2048, "outputs": 2048,
         "rank": 64, "bias": True, "keep": False, "dtype": "f32"},
        # q, k and v of one 4096-wide layer with the rotary step, 8192 packed tokens.
        {"name": "qkv-group", "kind": "qkv", "rows": 8192, "inputs": 4096, "heads": 32, "head_dim": 128,
         "rank": 256, "keep": True},
        # The SwiGLU block that keeps its intermediates (the usual training step), ragged batch.
        {"name": "mlp-cached", "kind": "mlp", "rows": 4001, "inputs": 2048, "inner": 8192, "rank": 256,
         "cache": True},
        # A whole decoder layer over three packed records, recomputing its MLP intermediates.
        {"name": "decoder-layer", "kind": "layer", "records": "1411,806,1204", "inputs": 2048, "heads": 16,
         "inner": 8192, "rank": 256},
        # Head product and weighted cross-entropy over the supervised part of a batch.
        {"name": "projection-loss", "kind": "loss", "rows": 2048, "supervised": 1500, "inputs": 2048,
         "vocab": 49152, "budget": 128, "scattered": False},
        # The optimizer over the adapters of four layers (d 2048, inner 8192, rank 256).
        {"name": "adamw-step", "kind": "adamw", "layers": 4, "inputs": 2048, "inner": 8192, "rank": 256},
        # Decoding a large weight (export, merging, a dense consumer).
        {"name": "nf4-decode", "kind": "decode", "outputs": 8192, "inputs": 8192, "storage": "bf16"},
        # Encoding a weight at load time (install_nf4's quantizer).
        {"name": "nf4-encode", "kind": "encode", "outputs": 11008, "inputs": 4096, "storage": "bf16"},
    ]


# ----------------------------------------------------------------------------- drawing cases
def _between(rng, low, high):
    """A whole number in [low, high], spread over its logarithm."""
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def _width(rng, low, high):
    """A feature count: a multiple of 64, or now and then only of 8."""
    unit = 8 if rng.random() < 0.15 else 64
    return max(low, _between(rng, low, high) // unit * unit)


def draw(rng):
    kind = rng.choice(["projection"] * 5 + ["qkv", "qkv", "mlp", "mlp", "layer", "loss", "adamw", "decode", "encode"])
    largest = work(next(c for c in listed() if c["name"] == "projection-long"))["flops"]
    while True:
        case = _draw_kind(rng, kind)
        if work(case)["flops"] <= 0.5 * largest:
            return case


def _draw_kind(rng, kind):
    rank = rng.choice([8, 16, 32, 64, 128, 256, 256])
    if kind == "projection":
        if rng.random() < 0.2:
            return {"kind": kind, "rows": _between(rng, 64, 2048), "inputs": _width(rng, 512, 4096),
                    "outputs": _width(rng, 512, 4096), "rank": rank, "bias": rng.random() < 0.5, "keep": False,
                    "dtype": "f32"}
        return {"kind": kind, "rows": _between(rng, 1, 16384), "inputs": _width(rng, 512, 24576),
                "outputs": _width(rng, 128, 24576), "rank": rank, "bias": rng.random() < 0.3,
                "keep": rng.random() < 0.7, "dtype": "bf16"}
    if kind == "qkv":
        heads = rng.choice([8, 12, 16, 24, 32])
        head_dim = rng.choice([64, 128])
        return {"kind": kind, "rows": _between(rng, 16, 8192), "inputs": heads * head_dim, "heads": heads,
                "head_dim": head_dim, "rank": rank, "keep": rng.random() < 0.7}
    if kind == "mlp":
        return {"kind": kind, "rows": _between(rng, 16, 8192), "inputs": _width(rng, 1024, 4096),
                "inner": _width(rng, 2048, 11008), "rank": rank, "cache": rng.random() < 0.6}
    if kind == "layer":
        records = [_between(rng, 17, 1500) for _ in range(rng.randint(1, 4))]
        heads = rng.choice([8, 16])
        return {"kind": kind, "records": ",".join(map(str, records)), "inputs": heads * 128, "heads": heads,
                "inner": _width(rng, 2048, 8192), "rank": rank}
    if kind == "loss":
        rows = _between(rng, 64, 4096)
        return {"kind": kind, "rows": rows, "supervised": rng.randint(max(1, rows // 4), rows),
                "inputs": _width(rng, 1024, 4096), "vocab": rng.choice([32000, 49152, 50257, 65536]),
                "budget": rng.choice([128, 128, 256]), "scattered": rng.random() < 0.4}
    if kind == "adamw":
        return {"kind": kind, "layers": rng.randint(1, 4), "inputs": _width(rng, 1024, 4096),
                "inner": _width(rng, 2048, 11008), "rank": rank}
    return {"kind": kind, "outputs": _width(rng, 512, 16384), "inputs": _width(rng, 512, 8192),
            "storage": rng.choice(["bf16", "bf16", "f16", "f32"])}


# ----------------------------------------------------------------------------- inputs
def _generator(seed):
    return torch.Generator(device=DEVICE).manual_seed(int(seed) & 0x7fffffffffffffff)


def _normal(g, *shape, std=1.0, dtype=torch.bfloat16):
    return (torch.randn(*shape, device=DEVICE, generator=g) * std).to(dtype)


def _fill_adapter(p, g):
    """Adapter values as training meets them: A at its initial spread, B away from zero."""
    k = p.lora_A.shape[1]
    with torch.no_grad():
        p.lora_A.copy_((torch.rand(p.lora_A.shape, device=DEVICE, generator=g) * 2 - 1) * (6 / k) ** 0.5)
        p.lora_B.copy_(torch.randn(p.lora_B.shape, device=DEVICE, generator=g) * 0.01)
        if p.bias is not None:
            p.bias.copy_(torch.randn(p.bias.shape, device=DEVICE, generator=g) * 0.1)


def _projection(inputs, outputs, rank, g, *, bias=False, dtype=torch.bfloat16):
    """A projection with an NF4 base quantized from ~N(0, 0.02)."""
    p = Projection(inputs, outputs, bias=bias, rank=rank, base_dtype=dtype, compute_dtype=dtype, device=DEVICE)
    p.install_nf4(_normal(g, outputs, inputs, std=0.02, dtype=dtype), DEVICE)
    _fill_adapter(p, g)
    return p


def _install(module, g):
    """NF4 bases and adapter values for every projection of a block built dense."""
    for p in module.modules():
        if isinstance(p, Projection):
            p.install_nf4(_normal(g, *p.weight.shape, std=0.02), DEVICE)
            _fill_adapter(p, g)


def _adapters(modules):
    return [t for p in modules for t in (p.lora_A, p.lora_B)]


def _records(case):
    bounds, start = [], 0
    for size in map(int, case["records"].split(",")):
        bounds.append((start, start + size))
        start += size
    return bounds, start


def _adapter_shapes(case):
    d, inner, r = case["inputs"], case["inner"], case["rank"]
    pairs = [(d, d), (d, 128), (d, 128), (d, d), (d, inner), (d, inner), (inner, d)]
    return [shape for _ in range(case["layers"]) for k, n in pairs for shape in ((r, k), (n, r))]


def prepare(case, seed):
    kind, g = case["kind"], _generator(seed)
    state = {"case": case}
    if kind == "projection":
        dtype = DTYPES[case["dtype"]]
        p = _projection(case["inputs"], case["outputs"], case["rank"], g, bias=case["bias"], dtype=dtype)
        state.update(modules=[p], x=_normal(g, case["rows"], case["inputs"], dtype=dtype).requires_grad_(True),
                     dy=[_normal(g, case["rows"], case["outputs"], dtype=dtype)])
    elif kind == "qkv":
        d, hd, rows = case["inputs"], case["head_dim"], case["rows"]
        config = DecoderConfig(hidden_size=d, num_attention_heads=case["heads"], head_dim=hd)
        # positions restart at a record boundary, as packed batches do
        positions = record_positions([(0, rows - rows // 3), (rows - rows // 3, rows)], DEVICE)
        cosine, sine = rotary_values(positions, config, torch.bfloat16)
        modules = [_projection(d, n, case["rank"], g, bias=True) for n in (case["heads"] * hd, hd, hd)]
        state.update(modules=modules, x=_normal(g, rows, d).requires_grad_(True), rotary=(cosine, sine, hd),
                     dy=[_normal(g, rows, n) for n in (case["heads"] * hd, hd, hd)])
    elif kind == "mlp":
        block = MLP(case["inputs"], case["inner"], rank=case["rank"], device=DEVICE)
        _install(block, g)
        state.update(block=block, modules=[block.gate_proj, block.up_proj, block.down_proj],
                     x=_normal(g, case["rows"], case["inputs"]).requires_grad_(True),
                     residual=_normal(g, case["rows"], case["inputs"]), dy=[_normal(g, case["rows"], case["inputs"])])
    elif kind == "layer":
        records, total = _records(case)
        config = DecoderConfig(hidden_size=case["inputs"], num_attention_heads=case["heads"],
                               intermediate_size=case["inner"])
        layer = Layer(config, rank=case["rank"], device=DEVICE)
        _install(layer, g)
        with torch.no_grad():
            for norm in (layer.input_layernorm, layer.post_attention_layernorm):
                norm.weight.copy_(_normal(g, case["inputs"], std=0.1) + 1)
        cosine, sine = rotary_values(record_positions(records, DEVICE), config, torch.bfloat16)
        attn, mlp = layer.self_attn, layer.mlp
        state.update(layer=layer, records=records, trig=(cosine, sine),
                     modules=[attn.q_proj, attn.k_proj, attn.v_proj, attn.o_proj, mlp.gate_proj, mlp.up_proj,
                              mlp.down_proj],
                     x=_normal(g, 1, total, case["inputs"]).requires_grad_(True),
                     dy=[_normal(g, 1, total, case["inputs"])])
    elif kind == "loss":
        rows, d = case["rows"], case["inputs"]
        count = case["supervised"]
        weights = torch.zeros(rows, device=DEVICE)
        if case["scattered"]:
            chosen = torch.randperm(rows, device=DEVICE, generator=g)[:count].sort().values
        else:
            chosen = torch.arange(rows - count, rows, device=DEVICE)
        weights[chosen] = 1.0
        # the selection is made where the batch is built, as the collating code does
        selection = slice(rows - count, rows) if not case["scattered"] else chosen
        state.update(x=_normal(g, rows, d).requires_grad_(True), head=_normal(g, case["vocab"], d, std=0.02),
                     targets=torch.randint(case["vocab"], (rows,), device=DEVICE, generator=g), weights=weights,
                     selection=selection)
    elif kind == "adamw":
        params = [torch.nn.Parameter(_normal(g, *shape, std=0.02, dtype=torch.float32))
                  for shape in _adapter_shapes(case)]
        for p in params:
            p.grad = _normal(g, *p.shape, std=1e-3, dtype=torch.float32)
        state.update(params=params, optimizer=FusedAdamW(params, lr=1e-4, betas=(0.9, 0.999), eps=1e-8,
                                                         weight_decay=0.01))
    else:
        weight = _normal(g, case["outputs"], case["inputs"], std=0.02, dtype=DTYPES[case["storage"]])
        if kind == "encode":
            state.update(weight=weight)
        else:
            packed, quantized = quantize_nf4(weight)
            state.update(packed=packed, quantized=quantized)
    return state


# ----------------------------------------------------------------------------- one pass
def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "projection" or kind == "qkv":
        with projection_budget(BUDGET if case["keep"] else 0):
            outputs = project_group(tuple(state["modules"]), state["x"], rotary=state.get("rotary"))
        return (*outputs, *torch.autograd.grad(outputs, [state["x"], *_adapters(state["modules"])], state["dy"]))
    if kind == "mlp":
        out = state["block"](state["x"], residual=state["residual"], cache=case["cache"])
        return (out, *torch.autograd.grad(out, [state["x"], *_adapters(state["modules"])], state["dy"][0]))
    if kind == "layer":
        with projection_budget(BUDGET):
            out = state["layer"](state["x"], *state["trig"], state["records"])
        return (out, *torch.autograd.grad(out, [state["x"], *_adapters(state["modules"])], state["dy"][0]))
    if kind == "loss":
        loss = projection_loss(state["x"], state["head"], state["targets"], state["weights"],
                               token_budget=case["budget"], rows=state["selection"])
        return (loss, *torch.autograd.grad(loss, [state["x"]]))
    if kind == "adamw":
        state["optimizer"].step()
        return tuple(state["params"])
    if kind == "decode":
        return dequantize_nf4(state["packed"], state["quantized"], state["quantized"].dtype)
    packed, quantized = quantize_nf4(state["weight"])
    return packed, quantized.absmax, quantized.state2.absmax, quantized.offset


# ----------------------------------------------------------------------------- what a pass needs
def _projection_work(m, k, n, r, size, packed=NF4_BYTES):
    """Forward, dx, dA and dB of one projection: the weight and the adapters read once, x, dy
    read once, out, dx and both gradients written once."""
    return {"bytes": packed * k * n + 8 * r * (k + n) + size * 2 * m * (k + n),
            "flops": 2 * m * (2 * k * n + 3 * r * (k + n))}


def _sum_work(parts, **more):
    total = {"bytes": more.get("bytes", 0), "flops": more.get("flops", 0)}
    for part in parts:
        total["bytes"] += part["bytes"]
        total["flops"] += part["flops"]
    return {key: float(value) for key, value in total.items()}


def _mlp_work(m, d, inner, r):
    """The three projections, with the activations between them counted as inner traffic."""
    parts = [_projection_work(m, d, inner, r, 0), _projection_work(m, d, inner, r, 0),
             _projection_work(m, inner, d, r, 0)]
    return parts


def work(case):
    kind = case["kind"]
    if kind == "projection":
        size = 4 if case["dtype"] == "f32" else 2
        return _sum_work([_projection_work(case["rows"], case["inputs"], case["outputs"], case["rank"], size)])
    if kind == "qkv":
        m, d, hd, r = case["rows"], case["inputs"], case["head_dim"], case["rank"]
        widths = (case["heads"] * hd, hd, hd)
        # x and dx are shared by the group
        return _sum_work([_projection_work(m, d, n, r, 2) for n in widths], bytes=-2 * 2 * 2 * m * d)
    if kind == "mlp":
        m, d = case["rows"], case["inputs"]
        # x, the residual and dy in, out and dx back
        return _sum_work(_mlp_work(m, d, case["inner"], case["rank"]), bytes=2 * m * d * 5)
    if kind == "layer":
        records, m = _records(case)
        d, r = case["inputs"], case["rank"]
        attention = [_projection_work(m, d, n, r, 0) for n in (d, 128, 128, d)]
        # causal attention, forward (2 products) and backward (5 with its recompute)
        scores = sum((b - a) * (b - a + 1) // 2 for a, b in records)
        return _sum_work(attention + _mlp_work(m, d, case["inner"], r), bytes=2 * m * d * 4,
                         flops=2 * 7 * scores * 128 * case["heads"])
    if kind == "loss":
        m, d, v = case["supervised"], case["inputs"], case["vocab"]
        return {"bytes": float(2 * v * d + 4 * m * d), "flops": float(4 * m * d * v)}
    if kind == "adamw":
        n = sum(a * b for a, b in _adapter_shapes(case))
        return {"bytes": float(28 * n), "flops": float(14 * n)}
    n = case["outputs"] * case["inputs"]
    size = 4 if case["storage"] == "f32" else 2
    return {"bytes": float((NF4_BYTES + size) * n), "flops": float((2 if kind == "decode" else 4) * n)}


def tolerance(case):
    """About four times the distance of the results from their 64-bit values (`exact`)."""
    kind = case["kind"]
    if kind in ("decode", "encode"):
        return "exact"
    if kind == "projection" and case["dtype"] == "f32":
        return {"rel": 6e-6}
    if kind == "adamw":
        return {"rel": 2e-7}
    # bf16: 1.7e-3 per rounding; the group, the MLP and the layer pass through several in a row
    return {"rel": {"projection": 8e-3, "loss": 8e-3, "qkv": 1.2e-2, "mlp": 1.6e-2, "layer": 3.6e-2}[kind]}


# ----------------------------------------------------------------------------- 64-bit restatement
def _dense(packed, s):
    """The base weight that the NF4 state `s` stands for, rounded to its storage type, in float64."""
    packed = packed.detach().reshape(-1)
    codes = torch.stack((packed >> 4, packed & 15), 1).reshape(-1).long()
    count = s.absmax.numel()
    second = s.state2.absmax.repeat_interleave(256)[:count]
    scales = s.state2.code[s.absmax.long()] * second + s.offset
    values = s.code[codes] * scales.repeat_interleave(s.blocksize)[:codes.numel()]
    return values[:s.shape.numel()].reshape(s.shape).to(s.dtype).double()


class _Exact:
    """One projection in float64: out = x w^T + bias + (x a^T) b^T and its gradients, with the
    factors as the compute dtype holds them."""

    def __init__(self, p):
        self.w = _dense(p.quantized.weight, p.quantized.weight.quant_state)
        self.a, self.b = (t.detach().to(p.compute_dtype).double() for t in (p.lora_A, p.lora_B))
        self.bias = None if p.bias is None else p.bias.detach().double()

    def forward(self, x):
        self.x, self.xa = x, x @ self.a.T
        out = x @ self.w.T + self.xa @ self.b.T
        return out if self.bias is None else out + self.bias

    def backward(self, dy):
        low = dy @ self.b
        self.grads = [low.T @ self.x, dy.T @ self.xa]
        return dy @ self.w + low @ self.a


def _rotate(x, cosine, sine, head_dim, inverse=False):
    """GPT-J rotation of the first 2 * half channels of every head, in float64."""
    half = cosine.shape[-1]
    y = x.reshape(*x.shape[:-1], -1, head_dim).clone()
    c, s = cosine.double().reshape(-1, 1, half), sine.double().reshape(-1, 1, half)
    s = -s if inverse else s
    even, odd = y[..., 0:2 * half:2].clone(), y[..., 1:2 * half:2].clone()
    y[..., 0:2 * half:2] = even * c - odd * s
    y[..., 1:2 * half:2] = odd * c + even * s
    return y.reshape(x.shape)


def _exact_mlp(modules, x):
    gate, up, down = (_Exact(p) for p in modules)
    g, u = gate.forward(x), up.forward(x)
    sigma = torch.sigmoid(g)
    out = down.forward(g * sigma * u)

    def backward(dy):
        dh = down.backward(dy)
        dx = gate.backward(dh * u * sigma * (1 + g * (1 - sigma))) + up.backward(dh * g * sigma)
        return dx, gate.grads + up.grads + down.grads
    return out, backward


def _rms(x, weight, eps):
    rstd = torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + eps)
    return x * rstd * weight, rstd


def _rms_backward(dy, x, rstd, weight):
    normed, scaled = x * rstd, dy * weight
    return rstd * (scaled - normed * (scaled * normed).mean(-1, keepdim=True))


def _exact_attention(q, k, v, records):
    """Causal attention within each record; q [H, S, D], k and v [S, D]. Returns out and a
    function from d out to (dq, dk, dv)."""
    saved, outs = [], []
    for a, b in records:
        scores = (q[:, a:b] @ k[a:b].T) * (q.shape[-1] ** -0.5)
        mask = torch.ones(b - a, b - a, dtype=torch.bool, device=q.device).triu(1)
        probabilities = scores.masked_fill(mask, float("-inf")).softmax(-1)
        saved.append(probabilities)
        outs.append(probabilities @ v[a:b])

    def backward(dout):
        dq, dk, dv = torch.empty_like(q), torch.empty_like(k), torch.empty_like(v)
        for (a, b), p in zip(records, saved):
            d = dout[:, a:b]
            dv[a:b] = (p.transpose(1, 2) @ d).sum(0)
            dp = d @ v[a:b].T
            ds = p * (dp - (dp * p).sum(-1, keepdim=True)) * (q.shape[-1] ** -0.5)
            dq[:, a:b] = ds @ k[a:b]
            dk[a:b] = (ds.transpose(1, 2) @ q[:, a:b]).sum(0)
        return dq, dk, dv
    return torch.cat(outs, 1), backward


def _exact_layer(state):
    case, layer = state["case"], state["layer"]
    x, dy = state["x"].detach()[0].double(), state["dy"][0][0].double()
    cosine, sine = state["trig"]
    heads, total = case["heads"], x.shape[0]
    norms = [(n.weight.detach().double(), n.eps) for n in (layer.input_layernorm, layer.post_attention_layernorm)]
    q, k, v, o = (_Exact(p) for p in state["modules"][:4])
    normed, rstd = _rms(x, *norms[0])
    qs = _rotate(q.forward(normed), cosine, sine, 128).view(total, heads, 128).transpose(0, 1)
    ks = _rotate(k.forward(normed), cosine, sine, 128)
    mixed, attention_backward = _exact_attention(qs, ks, v.forward(normed), state["records"])
    y = o.forward(mixed.transpose(0, 1).reshape(total, -1)) + x
    normed2, rstd2 = _rms(y, *norms[1])
    out, mlp_backward = _exact_mlp(state["modules"][4:], normed2)
    out = out + y
    dn2, mlp_grads = mlp_backward(dy)
    d_y = dy + _rms_backward(dn2, y, rstd2, norms[1][0])
    dq, dk, dv = attention_backward(o.backward(d_y).view(total, heads, 128).transpose(0, 1))
    dq = _rotate(dq.transpose(0, 1).reshape(total, -1), cosine, sine, 128, inverse=True)
    dn = q.backward(dq) + k.backward(_rotate(dk, cosine, sine, 128, inverse=True)) + v.backward(dv)
    dx = d_y + _rms_backward(dn, x, rstd, norms[0][0])
    return (out[None], dx[None], *q.grads, *k.grads, *v.grads, *o.grads, *mlp_grads)


def exact(case, seed):
    kind = case["kind"]
    if kind == "encode":
        return None  # whole values: bytes, and scales that are inputs' own maxima
    state = prepare(case, seed)
    with torch.no_grad():
        if kind == "projection" or kind == "qkv":
            x = state["x"].detach().double()
            parts = [_Exact(p) for p in state["modules"]]
            outputs, dx, grads = [], None, []
            for index, (part, dy) in enumerate(zip(parts, state["dy"])):
                out, d = part.forward(x), dy.double()
                if kind == "qkv" and index < 2:
                    out = _rotate(out, *state["rotary"])
                    d = _rotate(d, *state["rotary"], inverse=True)
                outputs.append(out)
                grad = part.backward(d)
                dx = grad if dx is None else dx + grad
                grads += part.grads
            return (*outputs, dx, *grads)
        if kind == "mlp":
            out, backward = _exact_mlp(state["modules"], state["x"].detach().double())
            dx, grads = backward(state["dy"][0].double())
            return (out + state["residual"].double(), dx, *grads)
        if kind == "layer":
            return _exact_layer(state)
        if kind == "loss":
            x, head = state["x"].detach(), state["head"].double()
            dx, total = torch.zeros(x.shape, dtype=torch.float64, device=DEVICE), 0.0
            rows = torch.arange(len(x), device=DEVICE)[state["selection"]]
            for part in rows.split(512):
                scale = state["weights"][part].double()
                logits = x[part].double() @ head.T
                log_z = torch.logsumexp(logits, 1)
                picked = state["targets"][part]
                total = total + (scale * (log_z - logits.gather(1, picked[:, None])[:, 0])).sum()
                soft = torch.exp(logits - log_z[:, None])
                soft.scatter_add_(1, picked[:, None], -torch.ones_like(soft[:, :1]))
                dx[part] = (soft * scale[:, None]) @ head
            return (total, dx)
        if kind == "adamw":
            # the first step: both moments start at zero, so their corrected values are the
            # gradient and its square
            results = []
            for p in state["params"]:
                w, grad = p.detach().double(), p.grad.double()
                results.append(w * (1 - 1e-4 * 0.01) - 1e-4 * grad / (grad.abs() + 1e-8))
            return tuple(results)
        return _dense(state["packed"], state["quantized"])
