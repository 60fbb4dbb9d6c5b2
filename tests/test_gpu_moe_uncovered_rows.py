"""Tokens whose router leaves them fewer than top_k experts (masked logits, -inf): the repeated slot has no row among the experts'
segments, the layer's intermediate rows behind the last segment hold whatever was in memory, and nothing of it reaches the output."""

import pytest
import torch

import mlc_llm_amd as gq
from mlc_llm_amd import ops
from mlc_llm_amd.nn import MixtralMoE

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scheme", ["q4f16_1", "q4bf16_1", "q4f32_1"])
@pytest.mark.parametrize("tokens,experts,top_k", [(3, 8, 2), (40, 8, 2), (130, 8, 2), (33, 24, 4), (6000, 8, 2)])
def test_repeated_slots_add_nothing(scheme, tokens, experts, top_k):
    hidden, inter = 256, 512
    config = gq.QUANTIZATION[scheme]
    dtype = {"float16": torch.float16, "bfloat16": torch.bfloat16, "float32": torch.float32}[config.model_dtype]
    g = torch.Generator(device="cuda").manual_seed(tokens)
    m = MixtralMoE(hidden, inter, experts, top_k, config, device="cuda")
    full = {}
    for name, (n, k) in (("e1_e3", (2 * inter, hidden)), ("e2", (hidden, inter))):
        w = (torch.randn((experts, n, k), generator=g, device="cuda") * 0.05).to(dtype)
        layer = getattr(m, name)
        layer.q_weight.data, layer.q_scale.data = ops.quantize(w, 4, 32)
        full[name] = ops.dequantize(layer.q_weight.data, layer.q_scale.data, k, 4, 32).double()
    x = torch.randn((1, tokens, hidden), generator=g, device="cuda").to(dtype)
    gate = torch.randn((tokens, experts), generator=g, device="cuda").to(dtype)
    gate[::3, 1:] = float("-inf")  # every third token is left with expert 0 alone
    weights, ids, _, _, pos, indptr = ops.moe_route(gate, top_k)
    pos = pos.view(tokens, top_k)
    short = len(range(0, tokens, 3))
    assert (pos[::3, 0] >= 0).all() and (pos[::3, 1:] == -1).all()
    assert int(indptr[-1]) == tokens * top_k - short * (top_k - 1) and int(pos.max()) == int(indptr[-1]) - 1
    poison = [torch.full((tokens * top_k, n), float("nan"), dtype=dtype, device="cuda") for n in (hidden, inter, hidden) for _ in range(2)]
    del poison  # the next allocations of these sizes find NaN
    out = m(x, gate)[0].double()
    # float64, expert by expert, on the ids and weights of the router (which has tests of its own; the masked experts weigh nothing)
    assert (weights[::3, 1:] == 0).all()
    p = torch.zeros((tokens, experts), device="cuda", dtype=torch.float64).scatter_add_(1, ids.long(), weights.double())
    want = torch.zeros_like(out)
    for e in range(experts):
        y = x[0].double() @ full["e1_e3"][e].t().contiguous()
        y = torch.nn.functional.silu(y[:, :inter]) * y[:, inter:]
        want += p[:, e : e + 1] * (y @ full["e2"][e].t().contiguous())
    err = ((out - want).norm() / want.norm()).item()
    # the roundings of the layer's four steps in the model dtype (2^-11, 2^-9 each), weights among them; float32 sums
    assert err <= {torch.float16: 4 * 2.0 ** -11, torch.bfloat16: 4 * 2.0 ** -9, torch.float32: 1e-5}[dtype], err
