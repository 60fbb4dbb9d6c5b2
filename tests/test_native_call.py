"""The native call path of linear, linear_silu_mul and embedding_take against the Python route, which a tensor subclass takes:
the same bits on every form that both accept, the same refusals."""

import numpy as np
import pytest
import torch

import mlc_llm_amd as gq
from mlc_llm_amd import ops


class Plain(torch.Tensor):
    """A subclass: the native path declines it, the Python route takes it."""


def _weights(n, k, scheme, device, seed=0):
    config = gq.QUANTIZATION[scheme]
    g = torch.Generator().manual_seed(seed)
    dtype = {"float16": torch.float16, "bfloat16": torch.bfloat16, "float32": torch.float32}[config.model_dtype]
    words, groups = ops.num_storage(k, config.bits, config.group_size), ops.num_group(k, config.group_size)
    qw = torch.randint(-2**31, 2**31 - 1, (n, words), generator=g, dtype=torch.int32)
    if config.bits == 3:
        qw &= (1 << 30) - 1
    qs = (torch.rand((n, groups), generator=g) * 0.01 + 0.001).to(dtype)
    return config, dtype, qw.to(device), qs.to(device)


@pytest.mark.gpu
@pytest.mark.parametrize("scheme", ["q4f16_1", "q3f16_1", "q4bf16_1", "q4f32_1"])
@pytest.mark.parametrize("lead", [(1,), (2, 3), (40,), (), (0,)])
def test_native_and_python_routes_agree(scheme, lead):
    n, k = 96, 320
    config, dtype, qw, qs = _weights(n, k, scheme, "cuda")
    x = torch.randn((*lead, k), device="cuda", dtype=torch.float32).to(dtype)
    bias = torch.randn((n,), device="cuda").to(dtype)
    residual = torch.randn((*lead, n), device="cuda").to(dtype)
    native = gq._lib.native()
    args = (qw, qs, config.bits, config.group_size)
    for b in (None, bias):
        for r in (None, residual):
            for out_dtype in (torch.float16, torch.float32):
                for given in (False, True):
                    own = dtype if out_dtype == torch.float16 else out_dtype
                    outs = [torch.empty((*lead, n), dtype=own, device="cuda") if given else None for _ in range(2)]
                    assert native.linear(x, *args, b, out_dtype, None, r) is not None
                    got = ops.linear(x, *args, b, out_dtype, outs[0], r)
                    want = ops.linear(x.as_subclass(Plain), *args, b, out_dtype, outs[1], r)
                    assert got.dtype == want.dtype == own and got.shape == want.shape == (*lead, n)
                    assert got.requires_grad is False and (outs[0] is None or got.data_ptr() == outs[0].data_ptr())
                    assert torch.equal(got, want.as_subclass(torch.Tensor))
    got, want = ops.linear_silu_mul(x, *args), ops.linear_silu_mul(x.as_subclass(Plain), *args)
    assert got.dtype == dtype and got.shape == (*lead, n // 2) and torch.equal(got, want.as_subclass(torch.Tensor))
    ids = torch.randint(0, n, lead, device="cuda", dtype=torch.int32)
    got = ops.embedding_take(ids, qw, qs, k, config.bits, config.group_size)
    want = ops.embedding_take(ids.as_subclass(Plain), qw, qs, k, config.bits, config.group_size)
    assert got.shape == (*lead, k) and torch.equal(got, want.as_subclass(torch.Tensor))


@pytest.mark.gpu
def test_the_native_path_runs_on_the_current_stream():
    config, dtype, qw, qs = _weights(64, 256, "q4f16_1", "cuda")
    x = torch.randn((3, 256), device="cuda", dtype=dtype)
    want = ops.linear(x, qw, qs, 4, 32)
    side = torch.cuda.Stream()
    assert gq._lib.native().stream() == torch.cuda.current_stream().cuda_stream
    graph = torch.cuda.CUDAGraph()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        assert gq._lib.native().stream() == side.cuda_stream
        ops.linear(x, qw, qs, 4, 32)
    torch.cuda.current_stream().wait_stream(side)
    with torch.cuda.graph(graph):
        got = ops.linear(x, qw, qs, 4, 32)
    for _ in range(3):
        got.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(got, want)


@pytest.mark.gpu
def test_refusals_are_the_python_routes():
    config, dtype, qw, qs = _weights(64, 256, "q4f16_1", "cuda")
    x = torch.randn((3, 256), device="cuda", dtype=dtype)
    wide = torch.randn((256, 6), device="cuda", dtype=dtype).t()  # not contiguous
    bad = [((x.double(), qw, qs), {}, TypeError), ((wide, qw, qs), {}, ValueError), ((x[:, :248].contiguous(), qw[:, :-1], qs), {}, ValueError),
           ((x, qw, qs[:, :-1].contiguous()), {}, ValueError), ((x, qw.float(), qs), {}, TypeError), ((x, qw, qs.float()), {}, TypeError),
           ((x, qw, qs), {"bias": torch.zeros(63, device="cuda", dtype=dtype)}, ValueError),
           ((x, qw, qs), {"residual": torch.zeros((3, 63), device="cuda", dtype=dtype)}, ValueError),
           ((x, qw, qs), {"out_dtype": torch.int32}, TypeError), ((x.cpu(), qw, qs), {}, ValueError), ((x.tolist(), qw, qs), {}, TypeError)]
    for args, kw, error in bad:
        with pytest.raises(error):
            ops.linear(*args, 4, 32, **kw)
    with pytest.raises(gq._lib.Mi355gqError) as err:  # a scheme that the library itself refuses
        ops.linear(x, torch.zeros((64, 64), device="cuda", dtype=torch.int32), qs, 8, 32)
    assert "mi355gq_linear" in str(err.value) and err.value.code != gq._lib.OK and err.value.message
    off = torch.zeros(3 * 256 + 1, device="cuda", dtype=dtype)[1:].view(3, 256)  # 2-byte aligned activations
    with pytest.raises(gq._lib.Mi355gqError, match="aligned"):
        ops.linear(off, qw, qs, 4, 32)
    with pytest.raises(ValueError):
        ops.linear_silu_mul(x, qw[:63].contiguous(), qs[:63].contiguous(), 4, 32)


def test_the_native_path_declines_what_is_not_a_plain_gpu_tensor():
    config, dtype, qw, qs = _weights(64, 256, "q4f16_1", "cpu")
    x, ids = torch.zeros((3, 256), dtype=dtype), torch.zeros(3, dtype=torch.int32)
    native = gq._lib.native()
    for first in (x, None, 3, x.to("meta"), np.zeros((3, 256))):
        assert native.linear(first, qw, qs, 4, 32, None, torch.float16, None, None) is None
        assert native.linear_silu_mul(first, qw, qs, 4, 32) is None
        assert native.embedding_take(first, qw, qs, 256, 4, 32) is None
    assert native.linear(x, qw, qs) is None and native.embedding_take(ids, qw, qs, 256, 4, 32) is None
    with pytest.raises(ValueError, match="GPU"):
        ops.linear(x, qw, qs, 4, 32)
    with pytest.raises(ValueError, match="GPU"):
        ops.linear_silu_mul(x, qw, qs, 4, 32)


@pytest.fixture
def without_native(tmp_path, monkeypatch):
    """The package as it is where the extension module was not built, or was built for another torch."""
    def use(content):
        path = tmp_path / "_mi355gq_torch.so"
        if content is not None:
            path.write_bytes(content)
        monkeypatch.setattr(gq._lib, "TORCH_PATH", str(path))
        monkeypatch.setattr(gq._lib, "_TORCH", None)
        with pytest.warns(RuntimeWarning, match="Python route"):
            assert gq._lib.native() is None
        assert gq._lib.native() is None  # (warned of once)
    return use


@pytest.mark.parametrize("content", [None, b"not a shared object"])
def test_without_the_extension_the_python_route_decides(without_native, content):
    without_native(content)
    _, dtype, qw, qs = _weights(8, 64, "q4f16_1", "cpu")
    with pytest.raises((TypeError, ValueError, RuntimeError)):
        ops.linear(torch.zeros((1, 64), dtype=dtype), qw, qs, 4, 32)  # (not on a GPU)


@pytest.mark.gpu
@pytest.mark.parametrize("scheme", ["q4f16_1", "q4f32_1"])
def test_every_operator_works_without_the_extension(without_native, scheme):
    n, k = 96, 320
    config, dtype, qw, qs = _weights(n, k, scheme, "cuda")
    x = torch.randn((5, k), device="cuda").to(dtype)
    ids = torch.randint(0, n, (4,), device="cuda", dtype=torch.int32)
    indptr = torch.tensor([0, 2, 5], device="cuda", dtype=torch.int32)
    experts = (torch.stack([qw, qw]), torch.stack([qs, qs]))

    def run():
        q, s = ops.quantize(x, 4, 32)
        return [ops.linear(x, qw, qs, 4, 32), ops.linear_silu_mul(x, qw, qs, 4, 32), ops.embedding_take(ids, qw, qs, k, 4, 32), q, s,
                ops.dequantize(qw, qs, k, 4, 32), ops.moe_group_gemm(x, *experts, indptr, 4, 32), ops.take_rows(x, ids)]

    want = run()
    without_native(None)
    for got, w in zip(run(), want):
        assert torch.equal(got, w)


def test_build_leaves_the_extension_out_without_a_compiler(tmp_path, monkeypatch):
    import importlib.util
    import os
    spec = importlib.util.spec_from_file_location("mi355gq_build_test", os.path.join(os.path.dirname(gq._lib.LIB_PATH), os.pardir, "build.py"))
    build = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(build)
    stale = tmp_path / "_mi355gq_torch.so"
    stale.write_bytes(b"")
    monkeypatch.setattr(build, "TORCH_EXT", str(stale))
    monkeypatch.setattr(build.shutil, "which", lambda name: None)
    assert build.build_torch_ext() is None and not stale.exists()
