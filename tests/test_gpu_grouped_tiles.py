"""Row tiles of expert segments: a wave finds its tile's expert among 64 at a time, so expert counts around 64 and its multiples, empty
segments at the ends and in between, tiles that do not exist; the tile heights by rows per expert.  Against the float64 product of
the dequantised weights."""

import pytest
import torch

import mlc_llm_amd as gq
from mlc_llm_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("experts", [1, 63, 64, 65, 130])
@pytest.mark.parametrize("average", [22, 40, 70, 150])
def test_every_row_meets_its_expert(dtype, experts, average):
    n, k = 72, 768
    g = torch.Generator().manual_seed(experts * average)
    sizes = torch.randint(0, 2 * average, (experts,), generator=g)
    sizes[torch.rand((experts,), generator=g) < 0.2] = 0
    if experts > 1:
        sizes[0] = sizes[-1] = 0
        sizes[experts // 2] += max(0, average * experts - int(sizes.sum()))  # one long segment brings the average up
    else:
        sizes[0] = average
    indptr = torch.cat([torch.zeros(1, dtype=torch.int64), sizes.cumsum(0)])
    rows = int(indptr[-1])
    gd = torch.Generator(device="cuda").manual_seed(experts + average)
    w = (torch.randn((experts, n, k), generator=gd, device="cuda") * 0.05).to(dtype)
    qw, qs = ops.quantize(w, 4, 32)
    full = ops.dequantize(qw, qs, k, 4, 32).double()
    x = torch.randn((rows, k), generator=gd, device="cuda").to(dtype)
    want = torch.empty((rows, n), dtype=torch.float64, device="cuda")
    for e in range(experts):
        want[indptr[e]:indptr[e + 1]] = x[indptr[e]:indptr[e + 1]].double() @ full[e].t().contiguous()
    got = ops.moe_group_gemm(x, qw, qs, indptr.int().cuda(), 4, 32)
    # one rounding of the output and float32 sums (a wrong expert is off by its whole row)
    tol = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -9, torch.float32: 0}[dtype] + 1e-5
    err = (got.double() - want).norm(dim=1) / want.norm(dim=1)
    assert err.max().item() <= 2 * tol, gq._lib.last_kernel()  # (2: a row of 72 elements, where the bound is for the mean)
    assert torch.equal(got, ops.moe_group_gemm(x, qw, qs, indptr.cuda(), 4, 32))
    short = ops.moe_group_gemm(torch.cat([x, x[:5]]), qw, qs, indptr.int().cuda(), 4, 32)  # rows behind the last segment
    assert (short[rows:] == 0).all() and (short[:rows].double() - want).norm() <= 2 * tol * want.norm()


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("experts,n,k,rows", [
    (64, 176, 2048, 384), (64, 160, 2048, 384),  # N % 32 == 16: the mid-row kernel's blocks do not fit the fused form; 0: they do
    (16, 80, 2048, 64), (128, 48, 512, 600), (8, 112, 4096, 160), (64, 176, 1408, 300), (8, 98, 1024, 300), (64, 112, 768, 4000),
    (20, 64, 704, 80), (20, 64, 704, 1200),
])
def test_fused_expert_segments_equal_the_two_steps(dtype, experts, n, k, rows):
    g = torch.Generator(device="cuda").manual_seed(experts + n + k)
    qw, qs = ops.quantize((torch.randn((experts * n, k), generator=g, device="cuda") * 0.02).to(dtype), 4, 32)
    qw, qs = qw.view(experts, n, -1), qs.view(experts, n, -1)
    counts = torch.bincount(torch.randint(0, experts, (rows,), generator=torch.Generator().manual_seed(rows)), minlength=experts)
    indptr = torch.cat([torch.zeros(1, dtype=torch.int64), counts.cumsum(0)]).int().cuda()
    x = torch.randn((rows, k), generator=g, device="cuda").to(dtype)
    plain = ops.moe_group_gemm(x, qw, qs, indptr, 4, 32)
    kernel = gq._lib.last_kernel()
    fused = ops.moe_group_gemm(x, qw, qs, indptr, 4, 32, silu_mul_halves=True)
    assert torch.equal(fused, ops.silu_mul(plain)), (kernel, gq._lib.last_kernel())


@pytest.mark.parametrize("n,rows_per_expert,tile", [
    (2048, 3, "quad_kernel<"), (2048, 6, "gemm_pipe_kernel<4,32,128,"), (64, 6, "quad_kernel<"), (64, 8, "gemm_pipe_kernel<4,32,128,"),
    (64, 60, "gemm_pipe_kernel<4,128,128,"), (64, 110, "gemm_pipe_kernel<4,256,")])
@pytest.mark.parametrize("k", [704, 1408])
def test_rules_by_rows_per_expert_hold_for_a_short_k_and_a_small_stack(k, n, rows_per_expert, tile):
    experts = 20
    rows = experts * rows_per_expert
    g = torch.Generator(device="cuda").manual_seed(k + rows)
    qw, qs = ops.quantize((torch.randn((experts * n, k), generator=g, device="cuda") * 0.02).half(), 4, 32)
    x = torch.randn((rows, k), generator=g, device="cuda").half()
    indptr = (torch.arange(experts + 1, dtype=torch.int32) * rows_per_expert).cuda()
    y = ops.moe_group_gemm(x, qw.view(experts, n, -1), qs.view(experts, n, -1), indptr, 4, 32)
    assert tile in gq._lib.last_kernel(), gq._lib.last_kernel()
    w = ops.dequantize(qw, qs, k, 4, 32).double().view(experts, n, k)
    want = torch.cat([x[e * rows_per_expert:(e + 1) * rows_per_expert].double() @ w[e].t().contiguous() for e in range(experts)])
    # one rounding of the output, and (few-row kernel) of each weight that it does not make
    assert (y.double() - want).norm() <= (2 * 2.0 ** -11 + 1e-5) * want.norm()


@pytest.mark.parametrize("experts,rows,kernel", [
    (16, 64, "quad_kernel<"), (16, 128, "midrow_kernel<1,"), (16, 320, "midrow_kernel<2,"),  # up to 16 experts: 4 to 8, then to 24
    (17, 40, "midrow_kernel<1,"), (24, 192, "midrow_kernel<1,"), (25, 175, "midrow_kernel<1,"), (25, 176, "midrow_kernel<2,"),
])
def test_midrow_bounds_by_experts(experts, rows, kernel):
    n, k = 64, 1024
    g = torch.Generator(device="cuda").manual_seed(rows)
    qw, qs = ops.quantize((torch.randn((experts * n, k), generator=g, device="cuda") * 0.02).half(), 4, 32)
    x = torch.randn((rows, k), generator=g, device="cuda").half()
    cuts = torch.linspace(0, rows, experts + 1).int()
    y = ops.moe_group_gemm(x, qw.view(experts, n, -1), qs.view(experts, n, -1), cuts.cuda(), 4, 32)
    assert kernel in gq._lib.last_kernel(), gq._lib.last_kernel()
    w = ops.dequantize(qw, qs, k, 4, 32).double().view(experts, n, k)
    want = torch.cat([x[cuts[e]:cuts[e + 1]].double() @ w[e].t().contiguous() for e in range(experts)])
    assert (y.double() - want).norm() <= (2 * 2.0 ** -11 + 1e-5) * want.norm()  # (as above)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("experts,n,average,tile", [
    # (float16 keeps the 256-row form)
    (4, 64, 128, "4,128,128,"), (12, 1408, 128, "4,128,128,"), (12, 2048, 128, "4,256,128,"),  # a CU each, or not
    (12, 2048, 256, "4,128,128,"), (17, 2048, 128, "4,128,128,"),  # one round of pairs against two
    (16, 4096, 128, "4,256,256,"),
])
def test_tall_tiles_of_long_segments(dtype, experts, n, average, tile):
    k = 128
    g = torch.Generator(device="cuda").manual_seed(experts + n)
    rows = experts * average
    cuts = torch.linspace(0, rows, experts + 1).int()
    cuts[1:-1] += torch.randint(-60, 60, (experts - 1,), generator=torch.Generator().manual_seed(n))
    qw, qs = ops.quantize((torch.randn((experts * n, k), generator=g, device="cuda") * 0.02).to(dtype), 4, 32)
    x = torch.randn((rows, k), generator=g, device="cuda").to(dtype)
    y = ops.moe_group_gemm(x, qw.view(experts, n, -1), qs.view(experts, n, -1), cuts.cuda(), 4, 32)
    if dtype == torch.float16 and tile == "4,128,128,":
        tile = "4,256,128,"
    assert f"gemm_pipe_kernel<{tile}" in gq._lib.last_kernel(), gq._lib.last_kernel()
    w = ops.dequantize(qw, qs, k, 4, 32).double().view(experts, n, k)
    want = torch.cat([x[cuts[e]:cuts[e + 1]].double() @ w[e].t().contiguous() for e in range(experts)])
    assert (y.double() - want).norm() <= ((2.0 ** -11 if dtype == torch.float16 else 2.0 ** -9) + 1e-5) * want.norm()  # one rounding
