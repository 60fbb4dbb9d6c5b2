"""The mid-row kernel's K slices where K is not whole phases: every slice takes the same number of shares, the last one fewer."""
import numpy as np
import pytest
import torch

import mlc_llm_amd as gq
from mlc_llm_amd import ops
from oracle import gq_oracle as o
from test_gpu_parity import SCHEMES, assert_linear_ok, dev, seed_of

pytestmark = pytest.mark.gpu


# shares of 256 k in the slices: 9 + 8, 10 + 10, 15 + 14 + 14, 14 each
@pytest.mark.parametrize("k,slices", [(4352, 2), (5120, 2), (11008, 3), (14336, 4)])
@pytest.mark.parametrize("m", [5, 16, 17])  # one batch tile, a full one, two
def test_midrow_kernel_even_slices(m, k, slices):
    """Against the oracle: the tolerance of every linear test (the products are exact, sums in fp32, one rounding of the result)."""
    s, n = SCHEMES["q4f16_1"], 544
    rng = np.random.default_rng(seed_of("even-slices", m, k))
    qw = rng.integers(0, 2**32, (n, k // 8), dtype=np.uint32)
    qs = (rng.random((n, k // 32)) * 0.02 + 0.001).astype(np.float16)
    x = rng.standard_normal((m, k)).astype(np.float16)
    out = torch.empty((m, n), dtype=torch.float16, device="cuda")
    scratch = torch.empty(slices * m * n, dtype=torch.float32, device="cuda")
    dx, dqw, dqs = dev(x), dev(qw), dev(qs)
    gq._lib.set_option("gemv_variant", 10)
    try:
        gq._lib.call("mi355gq_linear", dx.data_ptr(), dqw.data_ptr(), dqs.data_ptr(), None, m, n, k, 4, 32, gq._lib.F16,
                     out.data_ptr(), scratch.data_ptr(), scratch.numel() * 4, ops._stream())
        kern = gq._lib.last_kernel()
    finally:
        gq._lib.set_option("gemv_variant", -1)
    assert kern.startswith("gq::midrow_kernel<") and f"slices={slices} " in kern, kern
    assert_linear_ok(out, o.linear_fp32(x, qw, qs, s), x, k, f"even slices {m}x{n}x{k} [{kern}]")


# one batch tile and more than one chunk of rounds (few workgroups): K of three, four and eight shares of sixteen groups, and as slices of five
# and of seven, eight, ... ; a ragged last tile; one and two such shares, which sixteen waves of eight groups take
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("n,k", [(2600, 512), (1312, 1024), (872, 1536), (648, 2048), (328, 4096), (552, 5120), (320, 18944)])
@pytest.mark.parametrize("m", [5, 16])
def test_midrow_kernel_eight_waves(dtype, m, n, k):
    """Eight waves of sixteen groups, against the float64 product of the quantised weights (which this kernel does not round): the
    result's own rounding, 2^-11 / 2^-8 at most and half of it root-mean-square at most, beside sums in fp32 of products around 1031 x."""
    g = torch.Generator(device="cuda").manual_seed(n + k + m)
    qw = torch.randint(-2**31, 2**31 - 1, (n, k // 8), device="cuda", dtype=torch.int32, generator=g)
    qs = (torch.rand((n, k // 32), device="cuda", generator=g) * 0.02 + 0.001).to(dtype)
    x = torch.randn((m, k), device="cuda", generator=g).to(dtype)
    q = torch.stack([(qw >> (4 * i)) & 15 for i in range(8)], -1).reshape(n, k).double() - 7
    ref = x.double() @ (q * qs.double().repeat_interleave(32, 1)).T
    out = torch.empty((m, n), dtype=dtype, device="cuda")
    scratch = torch.empty(5 * m * n, dtype=torch.float32, device="cuda")
    code = gq._lib.F16 if dtype == torch.float16 else gq._lib.BF16
    gq._lib.set_option("gemv_variant", 10)
    gq._lib.set_option("gemv_waves", 16)  # one workgroup per slice
    try:
        gq._lib.call("mi355gq_linear_dt", x.data_ptr(), qw.data_ptr(), qs.data_ptr(), None, m, n, k, 4, 32, code, code,
                     out.data_ptr(), scratch.data_ptr(), scratch.numel() * 4, ops._stream())
        kern = gq._lib.last_kernel()
    finally:
        gq._lib.set_option("gemv_variant", -1)
        gq._lib.set_option("gemv_waves", -1)
    assert kern.startswith("gq::midrow_kernel<1,16," if k >= 1536 else "gq::midrow_kernel<1,8,"), kern
    err = (out.double() - ref).norm() / ref.norm()
    assert err <= (2.0**-11 if dtype == torch.float16 else 2.0**-8), (kern, err)


# the same on expert segments, one workgroup per expert
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("n,k", [(1184, 512), (608, 1024), (608, 1536), (608, 2048), (288, 4096)])
def test_midrow_kernel_eight_waves_of_expert_segments(dtype, n, k):
    """An empty expert, one of a single row, one of a whole batch tile, one of two passes and one of three, the gather of the rows folded in, against
    the float64 products (tolerance: see above); the fused gate/up form against the two steps."""
    g = torch.Generator(device="cuda").manual_seed(n + k)
    cuts = [0, 1, 1, 17, 36, 76]
    qw = torch.randint(-2**31, 2**31 - 1, (5, n, k // 8), device="cuda", dtype=torch.int32, generator=g)
    qs = (torch.rand((5, n, k // 32), device="cuda", generator=g) * 0.02 + 0.001).to(dtype)
    xs = torch.randn((25, k), device="cuda", generator=g).to(dtype)
    rows = torch.randint(0, 25, (76,), device="cuda", dtype=torch.int32, generator=g)
    ip, words = torch.tensor(cuts, dtype=torch.int32, device="cuda"), qw.view(torch.uint32)
    gq._lib.set_option("gemv_variant", 10)
    gq._lib.set_option("gemv_waves", 16)
    try:
        y = ops.moe_experts(xs, rows, words, qs, ip, 4, 32)
        kern = gq._lib.last_kernel()
        fused = ops.moe_experts(xs, rows, words, qs, ip, 4, 32, silu_mul_halves=True)
        kern_fused = gq._lib.last_kernel()
    finally:
        gq._lib.set_option("gemv_variant", -1)
        gq._lib.set_option("gemv_waves", -1)
    want = "gq::midrow_kernel<1,16," if k >= 1536 else "gq::midrow_kernel<1,8,"
    assert kern.startswith(want) and kern_fused.startswith(want) and " chunks=1 " not in kern, (kern, kern_fused)
    assert torch.equal(fused, ops.silu_mul(y)), kern
    q = torch.stack([(qw >> (4 * i)) & 15 for i in range(8)], -1).reshape(5, n, k).double() - 7
    w, x = q * qs.double().repeat_interleave(32, 2), xs[rows.long()].double()
    ref = torch.cat([x[cuts[e]:cuts[e + 1]] @ w[e].T for e in range(5)])
    each = (y.double() - ref).norm(dim=1) / ref.norm(dim=1)
    assert each.max() <= (2.0**-11 if dtype == torch.float16 else 2.0**-8), (kern, each)


def test_default_kernel_of_a_large_expert_stack():
    """48 rows over 8 experts of 28672 x 4096: eight waves, a sample of the columns against the float64 products (tolerance: see above), the fused
    gate/up form against the two steps."""
    e, n, k = 8, 28672, 4096
    g = torch.Generator(device="cuda").manual_seed(48)
    cuts = [0, 3, 9, 9, 26, 30, 37, 42, 48]
    qw = torch.randint(-2**31, 2**31 - 1, (e, n, k // 8), device="cuda", dtype=torch.int32, generator=g)
    qs = (torch.rand((e, n, k // 32), device="cuda", generator=g) * 0.02 + 0.001).half()
    x = torch.randn((48, k), device="cuda", generator=g).half()
    ip, words = torch.tensor(cuts, dtype=torch.int32, device="cuda"), qw.view(torch.uint32)
    y = ops.moe_experts(x, None, words, qs, ip, 4, 32)
    kern = gq._lib.last_kernel()
    fused = ops.moe_experts(x, None, words, qs, ip, 4, 32, silu_mul_halves=True)
    assert kern.startswith("gq::midrow_kernel<1,16,") and gq._lib.last_kernel().startswith("gq::midrow_kernel<1,16,"), (kern, gq._lib.last_kernel())
    assert torch.equal(fused, ops.silu_mul(y)), kern
    cols = torch.cat([torch.tensor([0, n // 2, n - 1], device="cuda"), torch.randint(0, n, (100,), device="cuda", generator=g)])
    for i in range(e):
        q = torch.stack([(qw[i, cols] >> (4 * f)) & 15 for f in range(8)], -1).reshape(len(cols), k).double() - 7
        ref = x[cuts[i]:cuts[i + 1]].double() @ (q * qs[i, cols].double().repeat_interleave(32, 1)).T
        assert (y[cuts[i]:cuts[i + 1]][:, cols].double() - ref).norm() <= 2.0**-11 * ref.norm(), (kern, i)


# at most two tiles per wave: K of eight, sixteen and fifteen shares (one idle wave); as few tiles as the dispatch sends, two rounds filled to
# the last tile, one tile more (the walk with a ring)
@pytest.mark.parametrize("n,k,m,once", [(2048, 2048, 17, 2), (16384, 2048, 32, 2), (8192, 4096, 17, 2), (8224, 4096, 32, 0), (1120, 3840, 17, 2),
                                        (2752, 3840, 9, 1), (4096, 4096, 16, 1), (2048, 5632, 12, 1)])
def test_midrow_kernel_of_two_rounds(m, n, k, once):
    """The default dispatch, against the float64 product of the quantised weights (tolerance: see above); bias and residual with a float32
    result, where what is left are sums in fp32; the fused gate/up form against the two steps.  Rows of tiny activations (one sixteenth of
    them is no float16) are as exact as others, and a row with an infinity has infinities or NaN alone, as its products have."""
    g = torch.Generator(device="cuda").manual_seed(n + k + m)
    qw = torch.randint(-2**31, 2**31 - 1, (n, k // 8), device="cuda", dtype=torch.int32, generator=g)
    qs = (torch.rand((n, k // 32), device="cuda", generator=g) * 0.02 + 0.001).half()
    x, b, r = (torch.randn(shape, device="cuda", generator=g).half() for shape in ((m, k), (n,), (m, n)))
    x[1] *= 1e-4
    q = torch.stack([(qw >> (4 * i)) & 15 for i in range(8)], -1).reshape(n, k).double() - 7
    w = q * qs.double().repeat_interleave(32, 1)
    ref = x.double() @ w.T
    words = qw.view(torch.uint32)
    y = ops.linear(x, words, qs, 4, 32)
    kern = gq._lib.last_kernel()
    assert kern.startswith(f"gq::midonce_kernel<{once},") if once else kern.startswith("gq::midrow_kernel<2,"), kern
    plain = ops.linear(x, words, qs, 4, 32, None, torch.float32)
    y32 = ops.linear(x, words, qs, 4, 32, b, torch.float32, residual=r)
    fused = ops.linear_silu_mul(x, words, qs, 4, 32)
    err = (y.double() - ref).norm() / ref.norm()
    assert err <= 2.0**-11, (kern, err)
    each = (plain.double() - ref).norm(dim=1) / ref.norm(dim=1)
    assert each.max() <= 5e-6 + 1e-7 * k**0.5, (kern, each)
    want = ref + b.double() + r.double()
    err32 = (y32.double() - want).norm() / want.norm()
    assert err32 <= 5e-6 + 1e-7 * k**0.5, (kern, err32)
    assert torch.equal(fused, ops.silu_mul(y))
    x[2, 5] = float("inf")
    y = ops.linear(x, words, qs, 4, 32)
    expect = torch.where(w[:, 5] == 0, float("nan"), torch.sign(w[:, 5]) * float("inf")).half()
    assert torch.equal(torch.isnan(y[2]), torch.isnan(expect)) and torch.equal(torch.nan_to_num(y[2]), torch.nan_to_num(expect)), kern
    assert torch.isfinite(y[[0, 1] + list(range(3, m))]).all()


# a wave without a share of K, in every form: the walk with a ring (one batch tile, two, eight waves, phases, slices) and the two rounds
@pytest.mark.parametrize("dtype,m,n,k,form,kernel", [
    (torch.float16, 5, 6016, 3840, "", "gq::midrow_kernel<1,8,"), (torch.float16, 9, 2752, 3840, "", "gq::midonce_kernel<1,"),
    (torch.float16, 16, 7040, 3584, "", "gq::midrow_kernel<1,8,"), (torch.float16, 17, 1120, 3840, "", "gq::midonce_kernel<2,"),
    (torch.float16, 32, 8224, 3840, "", "gq::midrow_kernel<2,8,"), (torch.float16, 5, 552, 5120, "one workgroup", "gq::midrow_kernel<1,16,"),
    (torch.float16, 6, 544, 14336, "forced", "gq::midrow_kernel<1,8,"), (torch.float16, 7, 544, 4352, "no scratch", "gq::midrow_kernel<1,8,"),
    (torch.bfloat16, 9, 1120, 3840, "", "gq::midrow_kernel<1,8,"), (torch.bfloat16, 24, 544, 3840, "forced", "gq::midrow_kernel<2,8,"),
    (torch.float32, 5, 1120, 3840, "", "gq::midrow_kernel<1,8,"), (torch.float32, 3, 1120, 14336, "", "gq::midrow_kernel<1,8,")])
def test_midrow_kernel_idle_waves_load_nothing(dtype, m, n, k, form, kernel):
    """Such a wave multiplies by zeros, so only a value that zero times it shows can tell what it has loaded: an infinite scale in the last
    group of K of some rows, tiles beyond the first among them.  There x is positive and the weights are, so that the group's sum is, of every
    plane of a float32 x (which meet as rows of their own, each scaled): these results are infinities, not NaN, and the others finite."""
    g = torch.Generator(device="cuda").manual_seed(n + k + m)
    qw = torch.randint(-2**31, 2**31 - 1, (n, k // 8), device="cuda", dtype=torch.int32, generator=g)
    qs = (torch.rand((n, k // 32), device="cuda", generator=g) * 0.02 + 0.001).to(dtype)
    x = torch.randn((m, k), device="cuda", generator=g).to(dtype)
    rows = [3, 19, n // 2, n - 1]
    qs[rows, -1] = float("inf")
    qw[rows, -4:] |= torch.tensor(0x88888888 - 2**32, dtype=torch.int32, device="cuda")  # (eight at least in every field)
    x[:, -32:] = x[:, -32:].abs()
    y = torch.empty((m, n), dtype=dtype, device="cuda")
    scratch = torch.empty(5 * m * n, dtype=torch.float32, device="cuda")
    code = {torch.float16: gq._lib.F16, torch.bfloat16: gq._lib.BF16, torch.float32: gq._lib.F32}[dtype]
    if form:
        gq._lib.set_option("gemv_variant", 10)
    if form == "one workgroup":
        gq._lib.set_option("gemv_waves", 16)
    try:
        gq._lib.call("mi355gq_linear_dt", x.data_ptr(), qw.data_ptr(), qs.data_ptr(), None, m, n, k, 4, 32, code, code, y.data_ptr(),
                     scratch.data_ptr(), 0 if form == "no scratch" else scratch.numel() * 4, ops._stream())
        kern = gq._lib.last_kernel()
    finally:
        gq._lib.set_option("gemv_variant", -1)
        gq._lib.set_option("gemv_waves", -1)
    assert kern.startswith(kernel) and (form != "no scratch" or " phases=2 " in kern), kern
    assert (y[:, rows] == float("inf")).all(), (kern, y[:, rows])
    rest = torch.ones(n, dtype=torch.bool, device="cuda")
    rest[rows] = False
    assert torch.isfinite(y[:, rest]).all(), kern


# one workgroup, more rounds than its chunks hold evenly: 18 as 10 + 8 (eight waves), 10 as 6 + 4 (sixteen), 6 as 4 + 2 (two batch tiles)
@pytest.mark.parametrize("dtype,m,n,k", [(torch.float16, 7, 288, 4096), (torch.float16, 7, 160, 3840), (torch.float16, 24, 96, 4096),
                                         (torch.bfloat16, 16, 288, 4096), (torch.bfloat16, 24, 96, 4096), (torch.float32, 5, 160, 4096)])
def test_midrow_kernel_shorter_last_chunk(dtype, m, n, k):
    """Against the float64 product of the quantised weights (tolerance: see test_midrow_kernel_eight_waves; float32: sums in fp32), and the fused
    gate/up form against the two steps.  float32: a row with an infinity, which the kernel finds by the sums of the last round walked."""
    g = torch.Generator(device="cuda").manual_seed(n + k + m)
    qw = torch.randint(-2**31, 2**31 - 1, (n, k // 8), device="cuda", dtype=torch.int32, generator=g)
    qs = (torch.rand((n, k // 32), device="cuda", generator=g) * 0.02 + 0.001).to(dtype)
    x = torch.randn((m, k), device="cuda", generator=g).to(dtype)
    q = torch.stack([(qw >> (4 * i)) & 15 for i in range(8)], -1).reshape(n, k).double() - 7
    w = q * qs.double().repeat_interleave(32, 1)
    words, fused = qw.view(torch.uint32), None
    gq._lib.set_option("gemv_variant", 10)
    gq._lib.set_option("gemv_waves", 16)
    try:
        y = ops.linear(x, words, qs, 4, 32, None, dtype)
        kern = gq._lib.last_kernel()
        if dtype != torch.float32:
            fused = ops.linear_silu_mul(x, words, qs, 4, 32)
        else:
            x[2, 5] = float("inf")
            odd = ops.linear(x, words, qs, 4, 32, None, dtype)[2]
            x[2, 5] = 0
    finally:
        gq._lib.set_option("gemv_variant", -1)
        gq._lib.set_option("gemv_waves", -1)
    assert kern.startswith("gq::midrow_kernel<") and " chunks=2 " in kern, kern
    if fused is not None:
        assert torch.equal(fused, ops.silu_mul(y)), kern
        ref = x.double() @ w.T
        assert (y.double() - ref).norm() / ref.norm() <= (2.0**-11 if dtype == torch.float16 else 2.0**-8), kern
    else:
        expect = torch.where(w[:, 5] == 0, float("nan"), torch.sign(w[:, 5]) * float("inf")).float()
        assert torch.equal(torch.isnan(odd), torch.isnan(expect)) and torch.equal(torch.nan_to_num(odd), torch.nan_to_num(expect)), kern
        rows = [0, 1, 3, 4]
        ref = x[rows].double() @ w.T
        assert (y[rows].double() - ref).norm() / ref.norm() <= 1e-6, kern


# the default dispatch on both sides of its bounds: (kernel, rows, N, K), float16
_QUADREG, _QUAD, _GEMM, _SKINNY = "gq::quadreg_kernel<", "gq::quad_kernel<", "gq::gemm_pipe_kernel<", "gq::skinny_q4_"
_WALK, _WIDE, _WALK2 = "gq::midrow_kernel<1,8,", "gq::midrow_kernel<1,16,", "gq::midrow_kernel<2,8,"
_ONCE, _ONCE2 = "gq::midonce_kernel<1,", "gq::midonce_kernel<2,"
_DEFAULTS = [
    # 17..32 rows of a short K
    (_GEMM, 32, 16384, 256), (_GEMM, 17, 10208, 1024), (_ONCE2, 17, 10240, 1024), (_ONCE2, 32, 20480, 512), (_GEMM, 17, 20448, 512), (_ONCE2, 17, 25472, 1024),
    (_GEMM, 17, 25504, 1024), (_ONCE2, 17, 3296, 1280), (_GEMM, 17, 3264, 1280), (_WALK2, 24, 20480, 1280), (_GEMM, 32, 25504, 1536), (_WALK2, 17, 39328, 1280),
    (_ONCE2, 17, 2048, 2048), (_GEMM, 17, 2016, 2048), (_WALK2, 17, 25504, 1792), (_ONCE2, 24, 8192, 2304), (_GEMM, 17, 8224, 2304), (_GEMM, 32, 10912, 2304),
    (_WALK2, 32, 10944, 2304), (_GEMM, 17, 8992, 2560), (_WALK2, 17, 9024, 2560), (_WALK2, 17, 8608, 2816),
    # ... and as K slices
    (_WALK2, 17, 5120, 16384), (_GEMM, 17, 4096, 20480), (_WALK2, 32, 4128, 20480), (_GEMM, 17, 4096, 24576), (_WALK2, 17, 3072, 28672), (_WALK2, 32, 10240, 8192), (_GEMM, 32, 10208, 8192),
    # 5..8 rows of one phase of K
    (_WALK, 6, 4576, 2304), (_QUADREG, 6, 4544, 2304), (_WALK, 5, 4128, 2560), (_QUADREG, 5, 4096, 2560), (_WALK, 8, 4128, 3584), (_QUADREG, 8, 4096, 3584),
    (_WALK, 5, 6016, 3840), (_QUADREG, 6, 5984, 3840), (_WALK, 7, 4128, 3840), (_QUADREG, 7, 4096, 3840), (_WALK, 6, 21504, 4096), (_QUADREG, 8, 21472, 4096),
    (_WALK, 5, 24576, 4096), (_QUADREG, 7, 24608, 4096), (_QUADREG, 8, 28672, 4096), (_WALK, 8, 28704, 4096), (_WIDE, 6, 38400, 4096), (_WALK, 7, 43008, 2048), (_QUADREG, 7, 42976, 2048),
    (_WIDE, 5, 37888, 3584),
    # ... as K slices
    (_WALK, 5, 4928, 5120), (_QUADREG, 5, 4896, 5120), (_WALK, 7, 4800, 6144), (_QUADREG, 8, 4768, 6144), (_WALK, 5, 6176, 7680), (_QUADREG, 8, 6144, 7680),
    (_WIDE, 6, 32768, 8192), (_QUAD, 6, 32736, 8192), (_QUAD, 5, 4096, 10240), (_WALK, 8, 4128, 10240), (_WALK, 8, 4096, 10496),
    # ... where the quad-row kernel with x in LDS takes the matrices of many rows
    (_WALK, 8, 31744, 4864), (_QUAD, 5, 31776, 4864), (_WALK, 8, 32800, 4864), (_QUAD, 5, 40992, 4864), (_WIDE, 5, 45056, 5120), (_QUAD, 8, 51200, 5120), (_WIDE, 5, 31744, 5120), (_QUAD, 5, 31776, 5120),
    (_QUAD, 8, 32768, 7168), (_WIDE, 8, 32800, 7168), (_WIDE, 5, 32768, 7680), (_WIDE, 8, 53248, 6144), (_QUAD, 5, 53280, 6144),
    # 9..16 rows below 24 M weights, where a wave walks two rounds or the skinny kernel answers
    (_ONCE, 12, 8192, 2560), (_SKINNY, 12, 9216, 2560), (_ONCE, 9, 4096, 5632), (_SKINNY, 16, 4128, 5632), (_ONCE, 9, 17760, 768), (_SKINNY, 9, 17728, 768),
    (_ONCE, 9, 12768, 1024), (_SKINNY, 12, 12800, 1024), (_SKINNY, 9, 16384, 1024), (_ONCE, 12, 16416, 1024), (_ONCE, 13, 13312, 1024),
]


# ... bfloat16, where the bounds are others
_DEFAULTS_BF16 = [
    (_WALK, 5, 28672, 4096), (_QUADREG, 8, 28640, 4096), (_WIDE, 5, 40960, 6144), (_QUAD, 8, 40992, 6144), (_WIDE, 7, 45056, 6656), (_QUAD, 6, 32768, 6144),
    (_WIDE, 6, 32768, 6656), (_WIDE, 5, 61440, 6656), (_WALK, 5, 4128, 3840), (_WALK, 16, 2048, 2048), (_GEMM, 9, 2016, 2048), (_WALK, 12, 4928, 5120), (_GEMM, 12, 4896, 5120), (_GEMM, 17, 28672, 4096),
]


@pytest.mark.parametrize("kernel,m,n,k,dtype", [(*d, torch.float16) for d in _DEFAULTS] + [(*d, torch.bfloat16) for d in _DEFAULTS_BF16])
def test_default_kernel_at_the_bounds(kernel, m, n, k, dtype):
    """Which kernel answers, a sample of the columns against the float64 product of the quantised weights (tolerance: one rounding of the
    result and, for the kernels that multiply such weights, one of every weight), and the fused gate/up form against the two steps."""
    g = torch.Generator(device="cuda").manual_seed(n + k + m)
    qw = torch.randint(-2**31, 2**31 - 1, (n, k // 8), device="cuda", dtype=torch.int32, generator=g)
    qs = (torch.rand((n, k // 32), device="cuda", generator=g) * 0.02 + 0.001).to(dtype)
    x = torch.randn((m, k), device="cuda", generator=g).to(dtype)
    words = qw.view(torch.uint32)
    y = ops.linear(x, words, qs, 4, 32, None, dtype)
    kern = gq._lib.last_kernel()
    assert kern.startswith(kernel), kern
    cols = torch.cat([torch.tensor([0, 1, n // 2, n - 1], device="cuda"), torch.randint(0, n, (200,), device="cuda", generator=g)])
    q = torch.stack([(qw[cols] >> (4 * i)) & 15 for i in range(8)], -1).reshape(len(cols), k).double() - 7
    ref = x.double() @ (q * qs[cols].double().repeat_interleave(32, 1)).T
    assert (y[:, cols].double() - ref).norm() / ref.norm() <= 2 * (2.0**-11 if dtype == torch.float16 else 2.0**-8), kern
    assert torch.equal(ops.linear_silu_mul(x, words, qs, 4, 32), ops.silu_mul(y)), kern


# float32: one or two rows of a small matrix load their own x, and three or four where a wave has one tile and a quarter of the waves no share
# of a short K; others take it from LDS (whole and idle shares of K, K slices)
@pytest.mark.parametrize("m,n,k,own", [(2, 48, 256, True), (2, 1120, 3840, True), (1, 1024, 9216, True), (2, 3056, 4096, True), (2, 3072, 4096, False),
                                       (3, 1120, 3840, False), (1, 1376, 9216, False), (3, 240, 768, True), (4, 336, 1536, True),
                                       (3, 8192, 1280, True), (4, 8208, 1280, False), (4, 4096, 2816, True), (3, 4112, 2816, False),
                                       (4, 160, 3072, False), (3, 256, 2048, False), (5, 304, 2560, False)])
def test_float32_rows_that_load_their_own_x(m, n, k, own):
    """Against the float64 product of the quantised weights (sums in fp32), and a row with an infinity."""
    g = torch.Generator(device="cuda").manual_seed(n + k + m)
    qw = torch.randint(-2**31, 2**31 - 1, (n, k // 8), device="cuda", dtype=torch.int32, generator=g)
    qs = torch.rand((n, k // 32), device="cuda", generator=g) * 0.02 + 0.001
    x = torch.randn((m, k), device="cuda", generator=g)
    q = torch.stack([(qw >> (4 * i)) & 15 for i in range(8)], -1).reshape(n, k).double() - 7
    w = q * qs.double().repeat_interleave(32, 1)
    y = ops.linear(x, qw.view(torch.uint32), qs, 4, 32, None, torch.float32)
    kern = gq._lib.last_kernel()
    assert kern.startswith("gq::midrow_kernel<1,8,2,0,0,f32>") and kern.endswith(" own x") == own, kern
    ref = x.double() @ w.T
    assert (y.double() - ref).norm() / ref.norm() <= 1e-6, kern
    x[m - 1, 5] = float("inf")
    odd = ops.linear(x, qw.view(torch.uint32), qs, 4, 32, None, torch.float32)
    expect = torch.where(w[:, 5] == 0, float("nan"), torch.sign(w[:, 5]) * float("inf")).float()
    assert torch.equal(torch.isnan(odd[m - 1]), torch.isnan(expect)) and torch.equal(torch.nan_to_num(odd[m - 1]), torch.nan_to_num(expect)), kern
    assert torch.equal(odd[:m - 1], y[:m - 1]), kern


# ... and of expert segments, one tile per wave and few rows per expert: a row each, twice as many where a quarter of the waves idle, one row or tile too many
@pytest.mark.parametrize("rows,experts,n,k,own", [(4, 4, 256, 4096, True), (5, 4, 336, 3840, True), (6, 4, 176, 1792, False), (8, 4, 1056, 768, True),
                                                  (9, 4, 304, 1280, False), (32, 16, 144, 2304, True), (8, 8, 512, 4096, True), (8, 8, 528, 4096, False)])
def test_float32_expert_rows_that_load_their_own_x(rows, experts, n, k, own):
    """Against the float64 products of the quantised weights (sums in fp32); the last expert has no row, and a row has an infinity."""
    g = torch.Generator(device="cuda").manual_seed(n + k + rows)
    qw = torch.randint(-2**31, 2**31 - 1, (experts, n, k // 8), device="cuda", dtype=torch.int32, generator=g)
    qs = torch.rand((experts, n, k // 32), device="cuda", generator=g) * 0.02 + 0.001
    x = torch.randn((rows, k), device="cuda", generator=g)
    of = torch.sort(torch.randint(0, experts - 1, (rows,), device="cuda", generator=g))[0]
    ip = torch.zeros(experts + 1, dtype=torch.int32, device="cuda")
    ip[1:] = torch.cumsum(torch.bincount(of, minlength=experts), 0).int()
    y = ops.moe_experts(x, None, qw.view(torch.uint32), qs, ip, 4, 32)
    kern = gq._lib.last_kernel()
    assert kern.startswith("gq::midrow_kernel<1,8,2,0,0,f32>") and kern.endswith(" own x") == own, kern
    q = torch.stack([(qw >> (4 * i)) & 15 for i in range(8)], -1).reshape(experts, n, k).double() - 7
    w = (q * qs.double().repeat_interleave(32, 2))[of]
    ref = torch.stack([w[i] @ x[i].double() for i in range(rows)])
    assert ((y.double() - ref).norm(dim=1) / ref.norm(dim=1)).max() <= 1e-6, kern
    x[1, 5] = float("inf")
    odd = ops.moe_experts(x, None, qw.view(torch.uint32), qs, ip, 4, 32)
    expect = torch.where(w[1, :, 5] == 0, float("nan"), torch.sign(w[1, :, 5]) * float("inf")).float()
    assert torch.equal(torch.isnan(odd[1]), torch.isnan(expect)) and torch.equal(torch.nan_to_num(odd[1]), torch.nan_to_num(expect)), kern
    rest = [i for i in range(rows) if i != 1]
    assert torch.equal(odd[rest], y[rest]), kern
