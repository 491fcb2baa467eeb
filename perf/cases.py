"""The work that users of the quantized linears have them do, as timed cases.

The sizes are the talker's and the code predictor's (hidden 2048 / 1024, the ones bench.py
and the tests use); `draw` adds ragged ones.  The kinds of a case:

* ``step``     the talker's decode step: ``layers`` decoder layers through the layer helpers,
               captured per padded batch (PaddedGraphs), as a serving loop replays it;
* ``frame``    the code predictor's walk: 15 prefix forwards of 5 layers in one graph;
* ``prefill``  decoder layers over a prompt's rows, eager, through the layer helpers;
* ``linears``  a layer's four linears on given activations, eager or as a captured step;
* ``linear``   one eager call of one linear;
* ``load``     what load time does with a layer's linears: quantize and re-tile the weights.

Layers get their weights as a checkpoint would fill them and are converted by
``quantize_module`` (``calibrate=False``: the kernels' own choice at every row count, so
that a case's route does not depend on timings).  The attention between qkv_proj and o_proj
is the caller's; its stand-in is the query part of qkv.
"""

from __future__ import annotations

import os
import sys

import torch
from torch import nn

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "tts-inference_amd"))

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}
#: hidden size, fused qkv width, attention (query) width, MLP width
MODELS = {"talker": (2048, 4096, 2048, 6144), "predictor": (1024, 4096, 2048, 3072)}
EPS = 1e-6
#: the code predictor's prefix lengths of one frame
PREFIXES = range(2, 17)


def listed():
    return [
        # One stream of speech: the whole talker stack, one row; bound by launches and the weight stream.
        {"name": "talker_step_batch1", "kind": "step", "model": "talker", "layers": 28, "rows": 1, "dtype": "bf16",
         "method": "int8_weight_only"},
        # A few streams, padded from 7 to the captured batch of 8 (12 layers still pass the caches).
        {"name": "talker_step_batch7", "kind": "step", "model": "talker", "layers": 12, "rows": 7, "dtype": "bf16",
         "method": "int8_weight_only"},
        # A busy server: 27 streams padded to 32 rows, past the decode kernels' 16.
        {"name": "talker_step_batch27", "kind": "step", "model": "talker", "layers": 12, "rows": 27, "dtype": "bf16",
         "method": "int8_weight_only"},
        # The predictor's walk, run once a frame for each talker step: one stream, and five padded to 8.
        {"name": "predictor_frame_batch1", "kind": "frame", "model": "predictor", "layers": 5, "rows": 1,
         "dtype": "bf16", "method": "int8_weight_only"},
        {"name": "predictor_frame_batch5", "kind": "frame", "model": "predictor", "layers": 5, "rows": 5,
         "dtype": "bf16", "method": "int8_weight_only"},
        # The smallest call: one row through one linear of the predictor, eager.
        {"name": "linear_1row", "kind": "linear", "n": 1024, "k": 2048, "rows": 1, "dtype": "bf16", "bias": False,
         "method": "int8_weight_only"},
        # Prompts through two talker layers, eager, an odd number of rows.
        {"name": "prefill_layers_1003", "kind": "prefill", "model": "talker", "layers": 2, "rows": 1003,
         "dtype": "bf16", "method": "int8_weight_only"},
        # fp8 weight-only with fp16 activations: a batch of short prompts.
        {"name": "prefill_fp8wo_640", "kind": "linears", "model": "talker", "layers": 1, "rows": 640, "dtype": "fp16",
         "method": "fp8_weight_only", "graph": False},
        # Both W8A8 methods over long prompts; the last is the largest case.
        {"name": "prefill_int8_1500", "kind": "linears", "model": "talker", "layers": 1, "rows": 1500, "dtype": "bf16",
         "method": "int8", "graph": False},
        {"name": "prefill_fp8_2048", "kind": "linears", "model": "talker", "layers": 1, "rows": 2048, "dtype": "bf16",
         "method": "fp8", "graph": False},
        # W8A8 decode: the linears of eight layers, three streams padded to 4.
        {"name": "decode_fp8_batch3", "kind": "linears", "model": "talker", "layers": 8, "rows": 3, "dtype": "bf16",
         "method": "fp8", "graph": True},
        # Loading a model: one talker layer's linears.
        {"name": "load_layer", "kind": "load", "model": "talker", "layers": 1, "dtype": "bf16",
         "method": "int8_weight_only"},
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, round(lo * (hi / lo) ** rng.random())))


def draw(rng):
    kind = rng.choice(["step", "step", "frame", "prefill", "prefill", "linears", "linears", "linears", "linear",
                       "linear", "load"])
    dtype = rng.choice(["bf16", "bf16", "bf16", "fp16"])
    method = rng.choice(["int8_weight_only", "fp8_weight_only", "int8", "fp8"])
    if kind == "step":
        return {"kind": kind, "model": rng.choice(["talker", "talker", "predictor"]), "layers": rng.randint(1, 14),
                "rows": _log(rng, 1, 64), "dtype": dtype, "method": "int8_weight_only"}
    if kind == "frame":
        return {"kind": kind, "model": "predictor", "layers": rng.randint(3, 5), "rows": rng.randint(1, 8),
                "dtype": dtype, "method": "int8_weight_only"}
    if kind == "prefill":
        return {"kind": kind, "model": rng.choice(["talker", "talker", "predictor"]), "layers": 1,
                "rows": _log(rng, 17, 2048), "dtype": dtype, "method": "int8_weight_only"}
    if kind == "linears":
        graph = rng.random() < 0.4
        return {"kind": kind, "model": rng.choice(["talker", "predictor"]), "layers": rng.randint(2, 8) if graph else 1,
                "rows": _log(rng, 1, 64) if graph else _log(rng, 17, 2048), "dtype": dtype, "method": method,
                "graph": graph}
    if kind == "linear":
        return {"kind": kind, "n": _log(rng, 200, 12288), "k": 64 * _log(rng, 4, 96), "rows": _log(rng, 1, 2048),
                "dtype": dtype, "bias": rng.random() < 0.5, "method": method}
    return {"kind": kind, "model": rng.choice(["talker", "predictor"]), "layers": rng.randint(1, 3), "dtype": dtype,
            "method": method}


# ---- the layers ----------------------------------------------------------------------------


def _shapes(case):
    """(N, K) of the case's linears, layer by layer."""
    if case["kind"] == "linear":
        return [(case["n"], case["k"])]
    hidden, qkv, attn, inter = MODELS[case["model"]]
    return [(qkv, hidden), (hidden, attn), (2 * inter, hidden), (hidden, inter)] * case["layers"]


def _weight(case, seed, index, n, k):
    g = torch.Generator(device="cuda").manual_seed(seed * 1000 + index)
    return (torch.randn(n, k, generator=g, device="cuda") * 0.02).to(DTYPES[case["dtype"]])


def _norm_weight(case, seed, index):
    g = torch.Generator(device="cuda").manual_seed(seed * 1000 + 500 + index)
    hidden = MODELS[case["model"]][0]
    return (1 + 0.1 * torch.randn(hidden, generator=g, device="cuda")).to(DTYPES[case["dtype"]])


def _bias(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed * 1000 + 900)
    return torch.randn(case["n"], generator=g, device="cuda").to(DTYPES[case["dtype"]]) if case["bias"] else None


def _inputs(case, seed, *shape):
    g = torch.Generator(device="cuda").manual_seed(seed * 1000 + 999)
    return torch.randn(*shape, generator=g, device="cuda").to(DTYPES[case["dtype"]])


class Norm(nn.Module):
    def __init__(self, weight):
        super().__init__()
        self.weight = nn.Parameter(weight, requires_grad=False)
        self.eps = EPS

    def forward(self, x):
        return torch.nn.functional.rms_norm(x, (x.shape[-1],), self.weight, self.eps)


class Layer(nn.Module):
    """A decoder layer's modules, named as the helpers expect them."""

    def __init__(self, case, seed, index):
        from qtts_amd.layers import GatedMLP, LinearBase, MergedLinear

        super().__init__()
        hidden, qkv, attn, inter = MODELS[case["model"]]
        kw = {"dtype": DTYPES[case["dtype"]], "device": "cuda"}
        kv = (qkv - attn) // 2
        self.input_layernorm = Norm(_norm_weight(case, seed, 2 * index))
        self.qkv_proj = MergedLinear(hidden, [attn, kv, kv], **kw)
        self.o_proj = LinearBase(attn, hidden, **kw)
        self.post_attention_layernorm = Norm(_norm_weight(case, seed, 2 * index + 1))
        self.mlp = GatedMLP(hidden, inter, **kw)
        for i, linear in enumerate(self.linears()):
            linear.weight.data.copy_(_weight(case, seed, 4 * index + i, linear.out_features, linear.in_features))

    def linears(self):
        return [self.qkv_proj, self.o_proj, self.mlp.gate_up_proj, self.mlp.down_proj]


def _quantized(case, module):
    from qtts_amd import QuantConfig, build_method, quantize_module

    config = QuantConfig(method=case["method"], calibrate=False)
    quantize_module(module, build_method(config), config, case["kind"])
    return module


def _decoder(case, layers, h):
    """The layers' data flow; returns the hidden state and every layer's qkv."""
    from qtts_amd.layers import decoder

    attn = MODELS[case["model"]][2]
    qkvs = []
    for layer in layers:
        qkv = decoder.norm_linear(layer.input_layernorm, layer.qkv_proj, h)
        qkvs.append(qkv)
        h = decoder.linear_residual(layer.o_proj, qkv[..., :attn], h)
        h = decoder.norm_mlp_residual(layer.post_attention_layernorm, layer.mlp, h)
    return (h, *qkvs)


def _walk(case, layers, x):
    """The predictor's frame: every prefix of the code positions through the layers."""
    return tuple(_decoder(case, layers, x[:, :p].reshape(-1, x.shape[-1]))[0].view(x.shape[0], p, x.shape[-1])
                 for p in PREFIXES)


def prepare(case, seed):
    from qtts_amd.graphs import PaddedGraphs
    from qtts_amd.layers import LinearBase

    case = dict(case)
    kind, dtype = case["kind"], DTYPES[case["dtype"]]
    with torch.no_grad():
        if kind == "load":
            weights = [_weight(case, seed, i, n, k) for i, (n, k) in enumerate(_shapes(case))]
            return {"case": case, "weights": weights}
        if kind == "linear":
            linear = LinearBase(case["k"], case["n"], bias=case["bias"], dtype=dtype, device="cuda")
            linear.weight.data.copy_(_weight(case, seed, 0, case["n"], case["k"]))
            if case["bias"]:
                linear.bias.data.copy_(_bias(case, seed))
            return {"case": case, "module": _quantized(case, nn.ModuleList([linear])),
                    "x": _inputs(case, seed, case["rows"], case["k"])}
        layers = _quantized(case, nn.ModuleList(Layer(case, seed, i) for i in range(case["layers"])))
        state = {"case": case, "module": layers}
        hidden = MODELS[case["model"]][0]
        if kind == "step":
            state["x"] = _inputs(case, seed, case["rows"], hidden)
            state["graphs"] = PaddedGraphs(lambda x: _decoder(case, layers, x), (hidden,), dtype)
        elif kind == "frame":
            state["x"] = _inputs(case, seed, case["rows"], PREFIXES[-1], hidden)
            state["graphs"] = PaddedGraphs(lambda x: _walk(case, layers, x), (PREFIXES[-1], hidden), dtype,
                                           batch_sizes=(1, 2, 4, 8))
        elif kind == "prefill":
            state["x"] = _inputs(case, seed, case["rows"], hidden)
        else:  # linears
            linears = [linear for layer in layers for linear in layer.linears()]
            width = max(linear.in_features for linear in linears)
            x = _inputs(case, seed, case["rows"], width)
            if case["graph"]:  # one padded buffer; each linear reads its columns of it
                state["x"] = x
                state["graphs"] = PaddedGraphs(lambda v: tuple(lin(v[:, :lin.in_features]) for lin in linears),
                                               (width,), dtype)
            else:
                state["calls"] = [(linear, x[:, :linear.in_features].contiguous()) for linear in linears]
        if "graphs" in state:  # captured before serving starts
            state["graphs"].run(state["x"])
    return state


def run(state):
    case = state["case"]
    with torch.no_grad():
        if case["kind"] == "load":
            return _load(case, state["weights"])
        if case["kind"] == "linear":
            return state["module"][0](state["x"])
        if "graphs" in state:
            return state["graphs"].run(state["x"])
        if case["kind"] == "prefill":
            return _decoder(case, state["module"], state["x"])
        return tuple(linear(x) for linear, x in state["calls"])


def _load(case, weights):
    from qtts_amd import QuantConfig, build_method
    from qtts_amd.layers import LinearBase

    method = build_method(QuantConfig(method=case["method"], calibrate=False))
    out = []
    for weight in weights:
        layer = LinearBase(weight.shape[1], weight.shape[0], dtype=weight.dtype, device="meta")
        layer.weight = nn.Parameter(weight, requires_grad=False)
        method.process_weights(layer)
        buffers = dict(layer.named_buffers())
        out += [b.view(torch.int8) if b.element_size() == 1 else b for _, b in sorted(buffers.items())]
    return tuple(out)


# ---- what a pass cannot do without -----------------------------------------------------------


def _rows(case):
    return sum(case["rows"] * p for p in PREFIXES) if case["kind"] == "frame" else case.get("rows", 0)


def work(case):
    shapes, m = _shapes(case), _rows(case)
    codes = sum(n * k for n, k in shapes)
    scales = sum(n for n, _ in shapes) * (2 if case["method"] == "int8_weight_only" else 4)
    if case["kind"] == "load":
        return {"bytes": 2 * codes + codes + scales, "flops": 0}
    flops = 2 * m * codes
    if case["kind"] in ("linear", "linears"):
        rows = sum(2 * m * (n + k) for n, k in shapes)
    else:  # the hidden state in and out, every layer's qkv out (a frame: the hidden states of each prefix)
        hidden, qkv, _, _ = MODELS[case["model"]]
        first = case["rows"] * PREFIXES[-1] if case["kind"] == "frame" else m
        rows = 2 * hidden * (first + m) + (0 if case["kind"] == "frame" else 2 * m * qkv * case["layers"])
    return {"bytes": codes + scales + rows, "flops": flops}


def tolerance(case):
    if case["kind"] == "load":
        return "exact"  # codes and scales are the reference's, bit for bit
    if case["kind"] in ("linear", "linears"):
        if case["method"] == "int8":
            return "exact"  # integer sums and a fixed epilogue
        # one rounding of the sums to 16 bits: 1.7e-3 (bf16) or 2.1e-4 (fp16) off the exact value
        return {"rel": 7e-3 if case["dtype"] == "bf16" else 9e-4}
    # the roundings of each layer's activations travel through those that follow
    deep = min(case["layers"], 8) ** 0.5
    return {"rel": min(0.03, (1e-2 if case["dtype"] == "bf16" else 1.3e-3) * deep)}


# ---- the same in 64 bits -----------------------------------------------------------------------


def _dequantized(case, w):
    """The weight that the case's method stores, as it multiplies, in 64 bits (and its codes' scale)."""
    f = w.float()
    amax = f.abs().amax(1, keepdim=True).clamp_min(1e-12)
    if case["method"].startswith("int8"):
        scale = amax * torch.tensor(1.0 / 127.0, dtype=torch.float32, device=w.device)
        q = torch.round(f / scale).clamp(-127, 127)
        if case["method"] == "int8_weight_only":
            scale = scale.to(w.dtype)
    else:
        scale = amax * torch.tensor(1.0 / 448.0, dtype=torch.float32, device=w.device)
        q = (f / scale).to(torch.float8_e4m3fn)
    return q.double() * scale.double()


def _activation(case, x):
    """The activation that the case's method multiplies (per-token codes for W8A8), in 64 bits."""
    if case["method"].endswith("weight_only"):
        return x.double()
    amax = x.abs().amax(1, keepdim=True).clamp_min(1e-6)
    if case["method"] == "int8":  # every step in the activation dtype
        scale = (amax.float() * torch.tensor(1.0 / 127.0, dtype=torch.float32, device=x.device)).to(x.dtype)
        return torch.round((x.float() / scale.float()).to(x.dtype)).clamp(-127, 127).double() * scale.double()
    scale = amax.float() * torch.tensor(1.0 / 448.0, dtype=torch.float32, device=x.device)
    return (x.float() / scale).to(torch.float8_e4m3fn).double() * scale.double()


def _exact_decoder(case, seed, h):
    _, _, attn, inter = MODELS[case["model"]]

    def norm(v, index):
        return v * torch.rsqrt(v.square().mean(-1, keepdim=True) + EPS) * _norm_weight(case, seed, index).double()

    qkvs = []
    shapes = _shapes(case)
    for layer in range(case["layers"]):
        w = [_dequantized(case, _weight(case, seed, 4 * layer + i, *shapes[i])) for i in range(4)]
        qkv = norm(h, 2 * layer) @ w[0].t()
        qkvs.append(qkv)
        h = h + qkv[:, :attn] @ w[1].t()
        gate, up = (norm(h, 2 * layer + 1) @ w[2].t()).split([inter, inter], -1)
        h = h + (torch.nn.functional.silu(gate) * up) @ w[3].t()
    return (h, *qkvs)


def exact(case, seed):
    with torch.no_grad():
        if case["kind"] == "load":
            out = []
            for i, (n, k) in enumerate(_shapes(case)):
                w = _weight(case, seed, i, n, k).double()
                scale = w.abs().amax(1) / (127.0 if case["method"].startswith("int8") else 448.0)
                out += [scale.reshape(1, -1) if case["method"] == "fp8" else scale, None]  # buffers in name order
            return tuple(out)
        if case["kind"] == "linear":
            y = _activation(case, _inputs(case, seed, case["rows"], case["k"])) @ _dequantized(
                case, _weight(case, seed, 0, case["n"], case["k"])).t()
            return y + _bias(case, seed).double() if case["bias"] else y
        hidden = MODELS[case["model"]][0]
        if case["kind"] == "linears":
            shapes = _shapes(case)
            x = _inputs(case, seed, case["rows"], max(k for _, k in shapes))
            return tuple(_activation(case, x[:, :k]) @ _dequantized(case, _weight(case, seed, i, n, k)).t()
                         for i, (n, k) in enumerate(shapes))
        if case["kind"] == "frame":  # all prefixes' rows at once: rows do not meet in these layers
            x = _inputs(case, seed, case["rows"], PREFIXES[-1], hidden).double()
            h = torch.cat([x[:, :p].reshape(-1, hidden) for p in PREFIXES])
            out = _exact_decoder(case, seed, h)[0].split([case["rows"] * p for p in PREFIXES])
            return tuple(v.view(case["rows"], p, hidden) for v, p in zip(out, PREFIXES))
        return _exact_decoder(case, seed, _inputs(case, seed, case["rows"], hidden).double())
