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
    (1, 48, 14336, "midrow"), (3, 1000, 1280, "midrow"), (5, 257, 4096, "midrow"), (4, 144, 8448, "midrow"),
    (2, 1000, 1280, "chunks=4"),  # one workgroup, whose sums meet several times
])
def test_linear(kind, m, n, k, kernel):
    x, qw, qs, rng = _operands(m, n, k, m + n + k)
    KINDS[kind](x[m // 2], rng.choice(k, 2, replace=False))
    args = (_dev(x), _dev(qw), _dev(qs))
    gq._lib.set_option("gemv_waves", 16 if "chunks" in kernel else -1)
    try:
        y = ops.linear(*args, 4, 32)
    finally:
        gq._lib.set_option("gemv_waves", -1)
    assert kernel in gq._lib.last_kernel(), gq._lib.last_kernel()
    if k > 4096:  # without scratch: K in phases
        out = torch.empty_like(y)
        gq._lib.call("mi355gq_linear_dt", *(t.data_ptr() for t in args), None, m, n, k, 4, 32, gq._lib.F32, gq._lib.F32, out.data_ptr(),
                     None, 0, torch.cuda.current_stream().cuda_stream)
        assert "midrow_kernel<1,8,2,0,1" in gq._lib.last_kernel(), gq._lib.last_kernel()
        _check(out.double().cpu().numpy(), x, o.dequantize_dt(qw, qs, S, k, "float32").astype(np.float64), k, kind)
    _check(y.double().cpu().numpy(), x, o.dequantize_dt(qw, qs, S, k, "float32").astype(np.float64), k, kind)


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("experts,n,k,sizes,kernel", [
    (3, 144, 256, [40, 0, 33], "gemm_f32_kernel"), (4, 48, 512, [0, 1, 6, 4], "midrow"), (4, 32, 8448, [3, 0, 2, 1], "midrow"),
])
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


@pytest.mark.parametrize("kind", KINDS)
def test_expert_per_row(kind):
    experts, n, k = 5, 48, 8448
    x, qw, qs, rng = _operands(3, n, k, 3, experts)
    KINDS[kind](x[1], rng.choice(k, 2, replace=False))
    ids = np.array([[4, 0, 4]], dtype=np.int32)
    y = ops.moe_gemv(_dev(x), _dev(qw), _dev(qs), _dev(ids), 4, 32)
    assert "midrow" in gq._lib.last_kernel(), gq._lib.last_kernel()
    for i, e in enumerate(ids[0]):
        w = o.dequantize_dt(qw[e], qs[e], S, k, "float32").astype(np.float64)
        _check(y[i:i + 1].double().cpu().numpy(), x[i:i + 1], w, k, (kind, i))
