"""float32 models, activations at the ends of the type's range, through the kernels that cut x into bfloat16 planes: infinities, NaNs
(one whose payload lies in the low 16 bits alone, which a truncation to bfloat16 would turn into an infinity), values so large that
the unscaled integers of a group would overflow, and very small ones, each in one row among ordinary rows.

The reference is the float64 sum of the single products, so an infinity times a weight of zero is a NaN and any other is an
infinity with the product's sign.  Finite results: 1e-6 + 4e-8 sqrt(K) of the row's norm, the bar of the float32 kernels."""

import numpy as np
import pytest
import torch

import mlc_llm_amd as gq
from mlc_llm_amd import ops
from oracle import gq_oracle as o

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
S = o.SCHEMES["q4f16_1"]
LOW_NAN = np.frombuffer(np.uint32(0x7F800001).tobytes(), np.float32)[0]

KINDS = {
    "inf": lambda x, at: x.__setitem__(at[0], np.inf),
    "minus inf": lambda x, at: x.__setitem__(at[0], -np.inf),
    "both infinities": lambda x, at: (x.__setitem__(at[0], np.inf), x.__setitem__(at[1], -np.inf)),
    "nan": lambda x, at: x.__setitem__(at[0], np.nan),
    "low nan": lambda x, at: x.__setitem__(at[0], LOW_NAN),
    "large": lambda x, at: np.multiply(x, np.float32(2.0**124), out=x),
    "small": lambda x, at: np.multiply(x, np.float32(2.0**-100), out=x),
}


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a.view(np.int32) if a.dtype == np.uint32 else a)).to(DEV)


def _operands(m, n, k, seed, experts=None):
    rng = np.random.default_rng(seed)
    lead = (n,) if experts is None else (experts, n)
    ng = -(-k // 32)
    qw = rng.integers(0, 2**32, (*lead, 4 * ng), dtype=np.uint32)
    qs = (rng.random((*lead, ng)) * 0.01 + 1e-3).astype(np.float32)
    return rng.standard_normal((m, k)).astype(np.float32), qw, qs, rng


def _check(y, x, w, k, what):
    for r in range(len(x)):
        with np.errstate(invalid="ignore"):
            want = (w * x[r].astype(np.float64)).sum(axis=1)
        got = y[r]
        assert np.array_equal(np.isnan(got), np.isnan(want)), (what, r)
        inf = np.isinf(want)
        assert np.array_equal(got[inf], want[inf]), (what, r)
        ok = np.isfinite(want)
        assert np.isfinite(got[ok]).all(), (what, r)
        if ok.any():
            rel = np.linalg.norm(got[ok] - want[ok]) / np.linalg.norm(want[ok])
            assert rel <= 1e-6 + 4e-8 * np.sqrt(k), (what, r, rel)


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("m,n,k,kernel", [
    (12, 70, 40, "gemm_f32_kernel<32"), (40, 130, 1544, "gemm_f32_kernel<64"), (70, 300, 1024, "gemm_f32_kernel<128"),
    (16, 128, 4096, "gemm_f32_kernel<32"),  # K split over workgroups
])
def test_linear(kind, m, n, k, kernel):
    x, qw, qs, rng = _operands(m, n, k, m + n + k)
    KINDS[kind](x[m // 2], rng.choice(k, 2, replace=False))
    y = ops.linear(_dev(x), _dev(qw), _dev(qs), 4, 32)
    assert kernel in gq._lib.last_kernel(), gq._lib.last_kernel()
    _check(y.double().cpu().numpy(), x, o.dequantize_dt(qw, qs, S, k, "float32").astype(np.float64), k, kind)


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("experts,n,k,sizes,kernel", [(3, 144, 256, [40, 0, 33], "gemm_f32_kernel")])
def test_experts(kind, experts, n, k, sizes, kernel):
    m = sum(sizes)
    x, qw, qs, rng = _operands(m, n, k, m + n + k, experts)
    KINDS[kind](x[1], rng.choice(k, 2, replace=False))
    ip = np.concatenate([[0], np.cumsum(sizes)])
    y = ops.moe_group_gemm(_dev(x), _dev(qw), _dev(qs), _dev(ip.astype(np.int32)), 4, 32)
    assert kernel in gq._lib.last_kernel(), gq._lib.last_kernel()
    y = y.double().cpu().numpy()
    for e in range(experts):
        w = o.dequantize_dt(qw[e], qs[e], S, k, "float32").astype(np.float64)
        _check(y[ip[e]:ip[e + 1]], x[ip[e]:ip[e + 1]], w, k, (kind, e))
