"""The plain q4 GEMM beyond 64 rows: every tile that the cost model chooses between, whole and split along K, at sizes that leave
ragged rows, columns and K tiles, against the float64 product of the dequantised weights (whose packing has tests of its own)."""

import pytest
import torch

import mlc_llm_amd as gq
from mlc_llm_amd import ops

pytestmark = pytest.mark.gpu

# rows, N, K, tile, split along K
CASES = [(65, 256, 256, "64,128", False), (65, 256, 1000, "64,128", True), (65, 6000, 4096, "128", True),
         (333, 6000, 1000, "128,128", False), (513, 8200, 320, "128,256", False), (129, 4096, 4104, None, None), (160, 4096, 14336, "256,128", True),
         (257, 4100, 2048, None, None), (777, 4096, 8192, "256,128", None), (300, 28672, 1024, "256,256", False),
         (512, 28680, 512, "256,256", False), (1025, 2056, 4096, None, None),
         # a K shorter than a K tile, whose chunks past K are loaded from the row's start
         (65, 256, 8, None, False), (130, 200, 24, None, False), (300, 130, 56, None, False),
         # K up to 512: by rounds of workgroups where there are many (ragged rows on the 256-row tile as well), by the cost else
         (760, 12000, 360, "256,256,128,64,2,false,false", False), (1732, 3400, 64, "128,256", False), (2734, 2880, 80, "128,128", False), (300, 700, 360, "64,128", None),
         # several rounds of workgroups, in one launch (the last one in float16: in two)
         (300, 25000, 2048, None, None), (450, 37888, 1024, None, None), (1536, 12288, 1024, None, None)]


def _problem(dtype, m, n, k):
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    w = (torch.randn((n, k), generator=g, device="cuda") * 0.02).to(dtype)
    qw, qs = ops.quantize(w, 4, 32)
    x = torch.randn((m, k), generator=g, device="cuda").to(dtype)
    bias = torch.randn((n,), generator=g, device="cuda").to(dtype)
    residual = torch.randn((m, n), generator=g, device="cuda").to(dtype)
    want = x.double() @ ops.dequantize(qw, qs, k, 4, 32).double().t().contiguous()
    return x, qw, qs, bias, residual, want


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("m,n,k,tile,split", CASES)
def test_planned_tiles(dtype, m, n, k, tile, split):
    x, qw, qs, bias, residual, want = _problem(dtype, m, n, k)
    # one rounding of the output (2^-11, bfloat16 2^-9 of the element), and float32 sums of K terms (sqrt(K) 2^-24 of the norm)
    tol = (2.0 ** -11 if dtype == torch.float16 else 2.0 ** -9) + 1e-5
    full = want + bias.double() + residual.double()
    got = ops.linear(x, qw, qs, 4, 32, bias, residual=residual)
    kernel = gq._lib.last_kernel()
    assert (got.double() - full).norm() / full.norm() <= tol, kernel
    got32 = ops.linear(x, qw, qs, 4, 32, None, torch.float32)
    assert (got32.double() - want).norm() / want.norm() <= 1e-5, kernel
    need = gq._lib.lib().mi355gq_linear_dt_workspace_bytes(m, n, k, 4, 32, ops._MODEL_DTYPES[dtype])
    assert need <= 32 << 20
    if dtype == torch.float16:
        assert split is None or (need > 0) == split, need
        assert tile is None or f"gemm_pipe_kernel<4,{tile}," in kernel, kernel
    # without scratch: another plan, unsplit
    out = torch.empty((m, n), dtype=dtype, device="cuda")
    gq._lib.call("mi355gq_linear_dt", x.data_ptr(), qw.data_ptr(), qs.data_ptr(), bias.data_ptr(), m, n, k, 4, 32,
                 ops._MODEL_DTYPES[dtype], ops._MODEL_DTYPES[dtype], out.data_ptr(), None, 0, torch.cuda.current_stream().cuda_stream)
    full = want + bias.double()
    assert (out.double() - full).norm() / full.norm() <= tol, gq._lib.last_kernel()
    if n % 2 == 0:  # the fused gate/up form adds in the same order: the same bits as the two steps
        assert torch.equal(ops.linear_silu_mul(x, qw, qs, 4, 32), ops.silu_mul(ops.linear(x, qw, qs, 4, 32)))


# rows, N, K, the second launch: columns of the whole rounds first, the rest on a smaller tile, K split (float16 and bfloat16 alike)
TWO = [(130, 33036, 1544, "<4,64,128,", "split=4 after 32768 columns"),  # (sums read one at a time: N % 8 != 0)
       (130, 33544, 1544, "<4,64,128,", "split=4 after 32768 columns"), (385, 16400, 2048, "<4,64,128,", "split=8 after 16384 columns"),
       (320, 22016, 4096, "<4,64,128,", "split=8 after 21504 columns"), (4000, 8208, 1544, "<4,64,128,", "split=4 after 8192 columns")]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("m,n,k,tile,second", TWO)
def test_two_launches(dtype, m, n, k, tile, second):
    x, qw, qs, bias, residual, want = _problem(dtype, m, n, k)
    tol = (2.0 ** -11 if dtype == torch.float16 else 2.0 ** -9) + 1e-5  # (as above)
    for args, out_dtype, full, bar in (((bias,), dtype, want + bias.double(), tol),
                                       ((bias,), torch.float32, want + bias.double(), 1e-5),
                                       ((None,), dtype, want + residual.double(), tol)):
        given = residual.clone() if args[0] is None else None  # (in place)
        got = ops.linear(x, qw, qs, 4, 32, *args, out_dtype, out=given, residual=given)
        kernel = gq._lib.last_kernel()
        assert tile in kernel and kernel.endswith(second), kernel
        worst = ((got.double() - full).norm(dim=0) / full.norm(dim=0)).max()  # (a column that went elsewhere would show)
        assert worst <= 4 * bar, (kernel, worst)
    need = gq._lib.lib().mi355gq_linear_dt_workspace_bytes(m, n, k, 4, 32, ops._MODEL_DTYPES[dtype])
    split, head = int(second.split()[0][6:]), int(second.split()[2])
    assert need == split * m * (n - head) * 4


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("m,n,k,second", [(320, 22016, 4096, "split=8 after 21504 columns"), (130, 34560, 2048, "after 32768 columns")])
def test_fused_form_of_two_launches_adds_in_the_same_order(dtype, m, n, k, second):
    x, qw, qs, *_ = _problem(dtype, m, n, k)
    steps = ops.silu_mul(ops.linear(x, qw, qs, 4, 32))
    fused = gq._lib.native().linear_silu_mul(x, qw, qs, 4, 32)
    assert isinstance(fused, torch.Tensor) and second in gq._lib.last_kernel(), gq._lib.last_kernel()
    assert torch.equal(fused, steps)


@pytest.mark.parametrize("bits", [4, 3])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("m,n,k", [
    (4000, 8208, 1544), (1000, 8208, 1544),  # two launches, the second split
    (129, 2064, 4096), (300, 4098, 2048), (70, 130, 4096),  # split; halves that are no multiple of 32, odd ones
    (40, 8208, 1544), (64, 66, 4096), (33, 4112, 1000), (20, 72, 4096), (17, 4110, 2048), (32, 34, 1024),  # tiles of 64 and 32 rows
    (12, 16400, 4096), (9, 2064, 4096), (200, 8208, 1544), (300, 2, 4096),
])
def test_fused_form_of_any_half_adds_in_the_same_order(bits, dtype, m, n, k):
    """linear_silu_mul equals linear and silu_mul bit for bit also where the halves are not whole 32-column blocks and K is split."""
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    group = {4: 32, 3: 40}[bits]
    qw, qs = ops.quantize((torch.randn((n, k), generator=g, device="cuda") * 0.02).to(dtype), bits, group)
    x = torch.randn((m, k), generator=g, device="cuda").to(dtype)
    steps = ops.silu_mul(ops.linear(x, qw, qs, bits, group))
    fused = gq._lib.native().linear_silu_mul(x, qw, qs, bits, group)
    assert isinstance(fused, torch.Tensor), fused
    assert torch.equal(fused, steps), gq._lib.last_kernel()
