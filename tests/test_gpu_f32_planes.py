"""float32 models on the bfloat16 matrix cores: x enters as three bfloat16 planes (exactly), the weights as integers.  Edges of the
tiles of both kernels (five rows per pass, 16 weight rows per tile; 32 / 64 / 128 rows by 128 / 256 columns), partly filled last
groups, split K, expert segments and one expert per row, against the float64 product of the same operands.

Tolerance: the products are exact, so only float32 sums separate a result from the exact one: 1e-6 + 4e-8 sqrt(K) relative
(the bar of the other float32 kernels; observed about 1e-7)."""

import numpy as np
import pytest
import torch

import mlc_llm_amd as gq
from mlc_llm_amd import ops
from oracle import gq_oracle as o

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
S = o.SCHEMES["q4f16_1"]


def _case(m, n, k, seed, experts=None):
    rng = np.random.default_rng(seed)
    lead = (n,) if experts is None else (experts, n)
    ng = -(-k // 32)
    qw = rng.integers(0, 2**32, (*lead, 4 * ng), dtype=np.uint32)  # every field value, 15 included
    if k % 32:  # fields past K are zero, as the quantizer leaves them
        f = np.arange(32 * ng).reshape(4 * ng, 8) < k
        qw &= (f * (np.uint32(15) << (4 * np.arange(8, dtype=np.uint32)))).sum(axis=1).astype(np.uint32)
    qs = (rng.random((*lead, ng)) * 0.02 + 1e-3).astype(np.float32)
    # significands of 24 bits over a wide range of exponents, within a row too
    x = (rng.standard_normal((m, k)) * np.exp2(rng.integers(-12, 13, (m, k)))).astype(np.float32)
    return x, qw, qs, rng


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a.view(np.int32) if a.dtype == np.uint32 else a)).to(DEV)


def _close(y, ref, k, what):
    rel = np.linalg.norm(y.double().cpu().numpy() - ref) / np.linalg.norm(ref)
    assert rel <= 1e-6 + 4e-8 * np.sqrt(k), (what, rel)


@pytest.mark.parametrize("m,n,k,kernel", [
    (1, 48, 14336, "midrow"), (2, 16, 256, "midrow"), (3, 1000, 1280, "midrow"), (5, 257, 4096, "midrow"), (4, 144, 8448, "midrow"),
    (6, 16400, 4096, "midrow"), (10, 16400, 4096, "midrow"),
    (5, 100, 1000, "gemm"), (6, 129, 8, "gemm"), (5, 40, 16, "gemm"), (33, 130, 24, "gemm"), (31, 130, 1544, "gemm"), (32, 128, 4096, "gemm"), (33, 300, 360, "gemm"),
    (64, 128, 288, "gemm"), (65, 256, 4096, "gemm"), (128, 257, 64, "gemm"), (129, 16, 5632, "gemm"), (300, 520, 1544, "gemm"),
    (300, 22300, 1024, "split=4"),  # whole rounds of columns first, the K of the rest cut
])
def test_linear_f32_tiles(m, n, k, kernel):
    x, qw, qs, rng = _case(m, n, k, m * 7919 + n + k)
    bias, res = rng.standard_normal(n).astype(np.float32), rng.standard_normal((m, n)).astype(np.float32)
    w = o.dequantize_dt(qw, qs, S, k, "float32").astype(np.float64)
    ref = x.astype(np.float64) @ w.T
    args = (_dev(x), _dev(qw), _dev(qs), 4, 32)
    y = ops.linear(*args)
    assert kernel in gq._lib.last_kernel(), gq._lib.last_kernel()
    _close(y, ref, k, "plain")
    r = _dev(res)
    y = ops.linear(*args, bias=_dev(bias), residual=r, out=r)  # in place
    _close(y, ref + bias + res, k, "bias, residual")
    # without the caller's scratch (no split of K): the same tolerance
    out = torch.empty((m, n), dtype=torch.float32, device=DEV)
    gq._lib.call("mi355gq_linear_dt", args[0].data_ptr(), args[1].data_ptr(), args[2].data_ptr(), None, m, n, k, 4, 32,
                 gq._lib.F32, gq._lib.F32, out.data_ptr(), None, 0, torch.cuda.current_stream().cuda_stream)
    _close(out, ref, k, "no workspace")


def test_planes_hold_every_bit_of_x():
    """One activation per row that is not zero: the result is x * (q - 7) * s with three float32 roundings at most."""
    n, k = 64, 4096
    _, qw, qs, rng = _case(1, n, k, 5)
    for m in (4, 40):
        x = np.zeros((m, k), np.float32)
        at = rng.integers(0, k, m)
        x[np.arange(m), at] = np.frombuffer(rng.integers(0x30000000, 0x4fffffff, m, dtype=np.uint32).tobytes(), np.float32)
        w = o.dequantize_dt(qw, qs, S, k, "float32").astype(np.float64)
        y = ops.linear(_dev(x), _dev(qw), _dev(qs), 4, 32).double().cpu().numpy()
        ref = x.astype(np.float64) @ w.T
        assert np.abs(y - ref).max(where=ref != 0, initial=0) <= 4 * 2.0**-24 * np.abs(ref).max()
        assert (np.abs(y - ref) <= 4 * 2.0**-24 * np.abs(ref)).all()


@pytest.mark.parametrize("experts,n,k,sizes,kernel", [
    (4, 48, 512, [0, 1, 6, 4], "midrow"), (4, 32, 8448, [3, 0, 2, 1], "midrow"), (4, 40, 360, [5, 3, 0, 2], "gemm"),
    # K % 256 != 0 and up to two rows per expert (beyond K = 4096 one and a half): the dot-product kernel
    (4, 40, 360, [3, 1, 0, 2], "gemv_dt"), (4, 40, 360, [3, 1, 0, 4], "gemv_dt"), (8, 24, 4104, [3, 1, 0, 4, 0, 2, 1, 1], "gemv_dt"),
    (8, 24, 4104, [3, 1, 0, 4, 0, 3, 1, 1], "gemm"), (16, 1040, 4104, [1] * 9 + [0] * 7, "gemm"),  # (68 M weights)
    (16, 1040, 4104, [1] * 8 + [0] * 8, "gemv_dt"),
    (3, 144, 256, [40, 0, 33], "gemm"), (3, 300, 1544, [130, 1, 64], "gemm"), (2, 256, 64, [200, 150], "gemm"),
])
def test_experts_f32(experts, n, k, sizes, kernel):
    m = sum(sizes)
    x, qw, qs, _ = _case(m, n, k, m + n + k, experts)
    ip = np.concatenate([[0], np.cumsum(sizes)])
    y = ops.moe_group_gemm(_dev(x), _dev(qw), _dev(qs), _dev(ip.astype(np.int32)), 4, 32)
    assert kernel in gq._lib.last_kernel(), gq._lib.last_kernel()
    for e in range(experts):
        w = o.dequantize_dt(qw[e], qs[e], S, k, "float32").astype(np.float64)
        rows = slice(ip[e], ip[e + 1])
        if sizes[e]:
            _close(y[rows], x[rows].astype(np.float64) @ w.T, k, e)


@pytest.mark.parametrize("one_row", [True, False])
def test_expert_per_row_f32(one_row):
    experts, n, k = 5, 48, 8448
    x, qw, qs, _ = _case(1 if one_row else 3, n, k, 3, experts)
    ids = np.array([[4, 0, 4]], dtype=np.int32)
    y = ops.moe_gemv(_dev(x), _dev(qw), _dev(qs), _dev(ids), 4, 32)
    assert "midrow" in gq._lib.last_kernel(), gq._lib.last_kernel()
    for i, e in enumerate(ids[0]):
        w = o.dequantize_dt(qw[e], qs[e], S, k, "float32").astype(np.float64)
        _close(y[i], x[0 if one_row else i].astype(np.float64) @ w.T, k, i)


@pytest.mark.parametrize("m,n,k,kernel,with_scratch", [
    (8, 130, 4096, "midrow_kernel<1,8,2,0,0,f32>", "gemm_f32"), (10, 64, 1024, "midrow_kernel<1,8,2,0,0,f32>", "gemm_f32"),
    (6, 48, 14336, "midrow_kernel<1,8,2,0,", "gemm_f32"), (11, 130, 4096, "gemm_f32_kernel<32,128,32,32> split=1", "gemm_f32"),
    (3, 200, 1544, "gemv_dt_kernel<4,1,2> passes=2", "gemm_f32"), (6, 1032, 4104, "gemv_dt_kernel<4,1,2> passes=3", "gemm_f32"),
    (8, 64, 1000, "gemm_f32_kernel<32,128,32,32> split=1", "gemm_f32"), (4, 28680, 1544, "gemm_f32_kernel<32,128,32,32> split=1", "gemm_f32"),
    (4, 4104, 4104, "gemm_f32_kernel<32,128,32,32> split=1", "gemm_f32"), (5, 40, 264, "gemm_f32", "gemm_f32"),  # (wants no scratch)
])
def test_linear_f32_without_scratch(m, n, k, kernel, with_scratch):
    """Few rows whose split of K has no scratch: two passes of the mid-row kernel, passes of the dot-product kernel while they are
    the shorter, the unsplit GEMM otherwise."""
    x, qw, qs, rng = _case(m, n, k, m + n + k)
    bias, res = rng.standard_normal(n).astype(np.float32), rng.standard_normal((m, n)).astype(np.float32)
    ref = x.astype(np.float64) @ o.dequantize_dt(qw, qs, S, k, "float32").astype(np.float64).T + bias + res
    xd, wd, sd, bd, rd = map(_dev, (x, qw, qs, bias, res))
    y = ops.linear(xd, wd, sd, 4, 32, bias=bd, residual=rd)
    assert with_scratch in gq._lib.last_kernel(), gq._lib.last_kernel()
    _close(y, ref, k, "with scratch")
    need = gq._lib.lib().mi355gq_linear_dt_workspace_bytes(m, n, k, 4, 32, gq._lib.F32)
    small = torch.empty(max(need - 4, 16), dtype=torch.uint8, device=DEV)
    for ws, size in ((None, 0), (small.data_ptr(), max(need - 4, 0))):  # none, and less than asked for
        gq._lib.call("mi355gq_linear_residual_dt", xd.data_ptr(), wd.data_ptr(), sd.data_ptr(), bd.data_ptr(), rd.data_ptr(), m, n, k, 4, 32,
                     gq._lib.F32, gq._lib.F32, y.data_ptr(), ws, size, torch.cuda.current_stream().cuda_stream)
        assert kernel in gq._lib.last_kernel(), gq._lib.last_kernel()
        _close(y, ref, k, "without scratch")
