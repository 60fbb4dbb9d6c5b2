"""What the group-quantized path is timed on: the work that a program serving or converting a model hands to it.

Five kinds of pass, each through the public modules of `mlc_llm_amd` (eager calls, as `MixtralMoE` and a model's decoder layer
make them; no graph is captured):

* "linear"  one projection, the smallest call there is;
* "decode"  one step of a decoder's linears for a few token rows: embedding, `layers` x (qkv, o_proj + residual, gate_up with the
            activation folded in, down_proj + residual), output head in float32 logits.  Eight layers keep the weights of a pass
            far beyond every cache, as the 32 of a model do;
* "prefill" the four linears of one or two decoder layers over a chunk of prompt rows;
* "moe"     one mixture-of-experts layer (routing, both expert matmuls, the weighted sum);
* "pack"    weight conversion: quantize a matrix, and dequantize it again.

Weights are N(0, 0.02) quantised by the library itself, activations and router logits N(0, 1), ids uniform.  The normalisations and
the attention that stand between a model's linears are not on this path, so every layer gets inputs of its own.
"""

from __future__ import annotations

import os
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "mlc-llm_amd"))
import mlc_llm_amd as gq  # noqa: E402
from mlc_llm_amd import ops  # noqa: E402
from mlc_llm_amd.nn import MixtralMoE  # noqa: E402

_DTYPE = {"float16": torch.float16, "bfloat16": torch.bfloat16, "float32": torch.float32}
_BYTES = {"float16": 2, "bfloat16": 2, "float32": 4}


def _decoder(kind, name, scheme, rows, hidden, qkv, inter, vocab, layers, bias=False):
    return {"name": name, "kind": kind, "scheme": scheme, "rows": rows, "hidden": hidden, "qkv": qkv, "inter": inter,
            "vocab": vocab, "layers": layers, "bias": bias}


def _moe(name, scheme, tokens, hidden, inter, experts, top_k):
    return {"name": name, "kind": "moe", "scheme": scheme, "tokens": tokens, "hidden": hidden, "inter": inter,
            "experts": experts, "top_k": top_k}


def listed():
    return [
        # one o_proj-sized call for one token: what a launch and the way to it cost
        {"name": "linear_1row", "kind": "linear", "scheme": "q4f16_1", "rows": 1, "n": 4096, "k": 4096},
        # a single user's chat: one token through an 8B model's linears
        _decoder("decode", "decode_1row", "q4f16_1", 1, 4096, 6144, 14336, 128256, 8),
        # a few concurrent users (or drafted tokens): an odd number of rows
        _decoder("decode", "decode_7rows", "q4f16_1", 7, 4096, 6144, 14336, 128256, 8),
        # a server under load: continuous batching
        _decoder("decode", "decode_32rows", "q4f16_1", 32, 4096, 6144, 14336, 128256, 8),
        # the 3-bit scheme on a 7B model, one user
        _decoder("decode", "decode_1row_q3", "q3f16_1", 1, 4096, 12288, 11008, 32000, 8),
        # a float32 model (the scheme for hosts without half precision), a few users
        _decoder("decode", "decode_4rows_f32", "q4f32_1", 4, 4096, 6144, 14336, 128256, 2),
        # the default prefill chunk of a long prompt
        _decoder("prefill", "prefill_2048", "q4f16_1", 2048, 4096, 6144, 14336, 0, 2),
        # the ragged end of a prompt, a bfloat16 model with biased qkv
        _decoder("prefill", "prefill_777_bf16", "q4bf16_1", 777, 4096, 6144, 14336, 0, 1, True),
        # a prompt on a float32 model
        _decoder("prefill", "prefill_300_f32", "q4f32_1", 300, 4096, 6144, 14336, 0, 1),
        # mixture of experts: a small decode batch (every expert read), and a prompt chunk
        _moe("moe_16tokens", "q4f16_1", 16, 4096, 14336, 8, 2),
        _moe("moe_512tokens", "q4f16_1", 512, 4096, 14336, 8, 2),
        # converting one large matrix of a checkpoint
        {"name": "pack_gate_up", "kind": "pack", "scheme": "q4f16_1", "n": 28672, "k": 4096},
    ]


# (hidden, qkv, inter, vocab) of the decoders in this repository's tests and benchmark, a small generic one, and one whose sizes are
# multiples of nothing larger than 8
_DECODERS = [(4096, 6144, 14336, 128256), (4096, 12288, 11008, 32000), (5120, 15360, 13824, 32000), (8192, 10240, 28672, 32000),
             (3584, 4608, 18944, 32000), (2048, 2560, 5632, 32000), (1544, 2056, 4104, 20008)]
# (hidden, inter, experts, top_k)
_EXPERTS = [(4096, 14336, 8, 2), (2048, 1408, 64, 6), (3584, 2560, 64, 8), (2048, 768, 128, 8)]
_SCHEMES = ["q4f16_1"] * 6 + ["q3f16_1", "q4bf16_1", "q4f32_1", "q4f16_0"]


def _log(rng, low, high):
    return int(round(low * (high / low) ** rng.random()))


def draw(rng):
    kind = rng.choice(["linear", "decode", "decode", "decode", "prefill", "prefill", "moe", "moe", "pack"])
    scheme = rng.choice(_SCHEMES)
    if kind == "linear":
        return {"kind": kind, "scheme": scheme, "rows": _log(rng, 1, 64), "n": 8 * _log(rng, 128, 4096), "k": 8 * _log(rng, 128, 2048)}
    if kind == "pack":
        return {"kind": kind, "scheme": scheme, "n": _log(rng, 1000, 32000), "k": 8 * _log(rng, 128, 1024)}
    if kind == "moe":
        hidden, inter, experts, top_k = rng.choice(_EXPERTS)
        scheme = "q4f16_1" if scheme == "q4f16_0" else scheme  # expert stacks have no KN layout
        case = _moe("", scheme, _log(rng, 1, 256 if scheme == "q4f32_1" else 2048), hidden, inter, experts, top_k)
    else:
        hidden, qkv, inter, vocab = rng.choice(_DECODERS)
        bias = rng.random() < 0.3
        if kind == "decode":
            layers = max(1, min(8, int(2.0e9 / (hidden * (qkv + hidden + 3 * inter)))))
            if scheme == "q4f32_1":
                layers = min(layers, 2)
            case = _decoder(kind, "", scheme, _log(rng, 1, 64), hidden, qkv, inter, vocab, layers, bias)
        else:
            case = _decoder(kind, "", scheme, _log(rng, 65, 4096), hidden, qkv, inter, 0, 1, bias)
    del case["name"]
    # no drawn pass is more work than the largest listed one; a float32 pass is as long as a pass of eight times its work
    most = 0.9 * _size(listed()[6]) / (8 if scheme == "q4f32_1" else 1)
    rows = "tokens" if kind == "moe" else "rows"
    while _size(case) > most and case[rows] > 1:
        case[rows] = case[rows] * 3 // 4
    return case


def _size(case):
    w = work(case)
    return max(w["bytes"], w["flops"] / 50)


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _normal(shape, g, dtype, std=1.0):
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32 if dtype == torch.float32 else torch.float16).mul_(std).to(dtype)


def _fill(module, shape, config, g, transpose=False):
    """Quantised N(0, 0.02) weights of `shape` [..., N, K] into a quantised module's parameters."""
    w = _normal(shape, g, _DTYPE[config.model_dtype], 0.02)
    q_weight, q_scale = config.quantize_weight(w, output_transpose=transpose)
    module.q_weight.data, module.q_scale.data = q_weight, q_scale
    return module


def _linear(n, k, config, g, bias=False, out_dtype=None):
    m = gq.GroupQuantizeLinear(k, n, config, bias=bias, out_dtype=out_dtype, device="cuda")
    if bias:
        m.bias.data = _normal((n,), g, m.bias.dtype, 0.1)
    return _fill(m, (n, k), config, g, config.linear_weight_layout == "KN")


@torch.no_grad()
def prepare(case, seed):
    config, g = gq.QUANTIZATION[case["scheme"]], _generator(seed)
    dtype = _DTYPE[config.model_dtype]
    kind = case["kind"]
    state = {"kind": kind, "config": config}
    if kind == "linear":
        state["linear"] = _linear(case["n"], case["k"], config, g)
        state["x"] = _normal((case["rows"], case["k"]), g, dtype)
    elif kind in ("decode", "prefill"):
        hidden, inter, rows = case["hidden"], case["inter"], case["rows"]
        state["layers"] = [{
            "qkv": _linear(case["qkv"], hidden, config, g, case["bias"]),
            "o": _linear(hidden, hidden, config, g),
            "gate_up": _linear(2 * inter, hidden, config, g),
            "down": _linear(hidden, inter, config, g),
            "x": _normal((rows, hidden), g, dtype),  # the normalised hidden state
            "attn": _normal((rows, hidden), g, dtype),  # the attention's output
            "hidden": _normal((rows, hidden), g, dtype),  # the residual stream
        } for _ in range(case["layers"])]
        if case["vocab"]:
            state["embed"] = _fill(gq.GroupQuantizeEmbedding(case["vocab"], hidden, config, device="cuda"), (case["vocab"], hidden), config, g)
            state["head"] = _linear(case["vocab"], hidden, config, g, out_dtype="float32")
            state["ids"] = torch.randint(0, case["vocab"], (rows,), generator=g, device="cuda", dtype=torch.int32)
            state["x"] = _normal((rows, hidden), g, dtype)
    elif kind == "moe":
        m = MixtralMoE(case["hidden"], case["inter"], case["experts"], case["top_k"], config, device="cuda")
        _fill(m.e1_e3, (case["experts"], 2 * case["inter"], case["hidden"]), config, g)
        _fill(m.e2, (case["experts"], case["hidden"], case["inter"]), config, g)
        state["moe"] = m
        state["x"] = _normal((1, case["tokens"], case["hidden"]), g, dtype)
        state["gate"] = _normal((case["tokens"], case["experts"]), g, dtype)
    else:
        state["w"] = _normal((case["n"], case["k"]), g, dtype, 0.02)
    return state


def _projection(module, x, residual):
    """o_proj / down_proj: the residual rides in the matmul where the layout has that entry."""
    c = module.config
    if c.linear_weight_layout == "KN":
        return module(x) + residual
    return ops.linear(x, module.q_weight, module.q_scale, c.bits, c.group_size, residual=residual)


@torch.no_grad()
def run(state):
    kind = state["kind"]
    if kind == "linear":
        return state["linear"](state["x"])
    if kind == "moe":
        return state["moe"](state["x"], state["gate"])
    if kind == "pack":
        c, w = state["config"], state["w"]
        q_weight, q_scale = c.quantize_weight(w)
        return q_weight, q_scale, c.dequantize_weight(q_weight, q_scale, w.shape[-1])
    out = []
    if "embed" in state:
        out.append(state["embed"](state["ids"]))
    for layer in state["layers"]:
        out.append(layer["qkv"](layer["x"]))
        hidden = _projection(layer["o"], layer["attn"], layer["hidden"])
        act = layer["gate_up"].forward_silu_mul(hidden)
        out += [hidden, act, _projection(layer["down"], act, hidden)]
    if "head" in state:
        out.append(state["head"](state["x"]))
    return out


def _weight_bytes(config, n, k):
    groups = -(-k // config.group_size)
    return n * groups * (16 + _BYTES[config.model_dtype])


def work(case):
    config = gq.QUANTIZATION[case["scheme"]]
    e = _BYTES[config.model_dtype]
    kind = case["kind"]
    if kind == "pack":  # the matrix read, its codes and scales written, read and written again as a matrix
        n, k = case["n"], case["k"]
        return {"bytes": 2 * n * k * e + 2 * _weight_bytes(config, n, k), "flops": 0}
    if kind == "linear":
        n, k, rows = case["n"], case["k"], case["rows"]
        return {"bytes": _weight_bytes(config, n, k) + rows * (n + k) * e, "flops": 2 * rows * n * k}
    if kind == "moe":
        t, h, i, top_k = case["tokens"], case["hidden"], case["inter"], case["top_k"]
        # the experts that t tokens with top_k uniform choices each are expected to touch
        touched = case["experts"] * (1 - (1 - top_k / case["experts"]) ** t)
        per_expert = _weight_bytes(config, 2 * i, h) + _weight_bytes(config, h, i)
        return {"bytes": touched * per_expert + 2 * t * h * e + t * case["experts"] * e, "flops": 2 * t * top_k * 3 * h * i}
    h, q, i, rows, v = case["hidden"], case["qkv"], case["inter"], case["rows"], case["vocab"]
    shapes = [(q, h), (h, h), (2 * i, h), (h, i)]
    layer = sum(_weight_bytes(config, n, k) for n, k in shapes) + rows * e * (3 * h + q + h + 2 * i + h)
    total = {"bytes": case["layers"] * layer, "flops": case["layers"] * 2 * rows * sum(n * k for n, k in shapes)}
    if v:
        total["bytes"] += _weight_bytes(config, v, h) + rows * (h * e + v * 4) + rows * (4 + 2 * h * e)
        total["flops"] += 2 * rows * v * h
    return total


def tolerance(case):
    """Packed words, scales and dequantised values are exact.  A product's tolerance is two to four times the relative error against
    the float64 product of the dequantised weights, carried through the layer (float16 6e-4 to 8e-4, bfloat16 2e-3 to 4.4e-3,
    float32 7e-7 to 2.7e-6): the roundings of the model dtype in the outputs and, for float16 and bfloat16, in the dequantised
    weight; float32 sums of up to 28672 terms otherwise."""
    if case["kind"] == "pack":
        return "exact"
    return {"rel": {"float16": 2e-3, "bfloat16": 1e-2, "float32": 1e-5}[gq.QUANTIZATION[case["scheme"]].model_dtype]}
