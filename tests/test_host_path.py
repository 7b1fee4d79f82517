"""The native host path (aklr_amd._host) against the general Python path: what it serves, what it leaves to
that path, and that both give the same bits.

On the CPU: every call is left to the general path (no GPU tensor), whatever its arguments, and a call with
missing or unknown arguments raises what the Python function raises. On the GPU: over every form the ops
accept (layouts, scale modes, dtypes, bias, keyword and positional arguments, non-default streams), the
native path serves the call and its outputs equal the general path's bit for bit; over every form it does
not take, it returns None and the op's answer is the general path's (outputs or the same FallbackReason).
"""
from __future__ import annotations

import importlib.util
import sys
import warnings

import pytest
import torch

import aklr_amd
from aklr_amd import _build, _lib, layouts, workloads
from aklr_amd.dispatch import FallbackReason
from tests.helpers import say

DEV = "cuda:0"
FP8, E5M2 = torch.float8_e4m3fn, torch.float8_e5m2
NATIVE = {"quant_fp8": aklr_amd.per_group_quant_fp8, "quant_mxfp8": aklr_amd.per_group_quant_mxfp8,
          "quant_mxfp4": aklr_amd.dynamic_mxfp4_quant, "gemm_fp8": aklr_amd.gemm_a8w8_blockwise_scaled,
          "quant_gemm_fp8": aklr_amd.quant_gemm_a8w8_blockwise_scaled, "gemm_mxfp4": aklr_amd.gemm_a4w4_mxfp4}


@pytest.mark.parametrize("name", sorted(NATIVE))
def test_cpu_calls_are_left_to_the_general_path(native_lib, name):
    fn, op = _lib.host_function(name), NATIVE[name]
    x = torch.zeros((2, 128), dtype=torch.bfloat16)
    for args, kwargs in [((x,), {}), ((x, x, x, x), {}), ((x, x, x), {"operand_format": "none:none"}), ((), {}),
                         ((None, 1, "a", x), {}), ((x,) * 12, {}), ((x,), {"nope": 1}), ((x, x, x, x), {"a": x}),
                         ((x, x, x, x, (128, 128), "K", True, None, torch.bfloat16), {})]:
        assert fn(args, kwargs) is None
    assert op(*((x,) * (1 if name.startswith("quant_") and name != "quant_gemm_fp8" else 4))[: 3 if name == "quant_gemm_fp8" else 4]) \
        is FallbackReason.OUT_OF_CONTRACT
    with pytest.raises(TypeError):
        op()
    with pytest.raises(TypeError):
        op(x, nope=1)


class _Untouchable:
    def __getattr__(self, name):
        raise RuntimeError(f"{name} was asked for")


@pytest.mark.parametrize("name", sorted(NATIVE))
@pytest.mark.parametrize("kind", ["proxy", "untouchable"])
def test_what_is_no_tensor_is_refused_without_raising(name, kind):
    """A tracer's stand-in, or any object, answers no question that the plan would not ask."""
    graph = torch.fx.Graph()
    x = torch.fx.Proxy(graph.placeholder("x"), torch.fx.Tracer()) if kind == "proxy" else _Untouchable()
    count = {"quant_gemm_fp8": 3}.get(name, 1 if name.startswith("quant_") else 4)
    assert NATIVE[name](*(x,) * count) is FallbackReason.OUT_OF_CONTRACT
    assert NATIVE[name].serving(*(x,) * count) is FallbackReason.OUT_OF_CONTRACT


def _not_loading(monkeypatch):
    monkeypatch.delattr(aklr_amd, "_host", raising=False)
    monkeypatch.setitem(sys.modules, "aklr_amd._host", None)
    monkeypatch.setattr(_lib, "_host_missing", False)


def test_an_extension_that_does_not_load_leaves_the_general_path(native_lib, monkeypatch):
    _not_loading(monkeypatch)
    with pytest.warns(RuntimeWarning, match="_host"):
        assert _lib.host_function("quant_fp8") is None
    with warnings.catch_warnings():
        warnings.simplefilter("error")  # once
        assert _lib.host_function("gemm_fp8") is None


def test_the_extension_refuses_another_torch(native_lib, monkeypatch):
    spec = importlib.util.spec_from_file_location("another._host", _build.HOST_PATH)
    monkeypatch.setattr(torch, "__version__", "1.0.0")
    with pytest.raises(ImportError, match="built with torch"):
        importlib.util.module_from_spec(spec)


@pytest.mark.gpu
def test_ops_serve_without_the_extension(monkeypatch):
    say("host path without the extension")
    from aklr_amd import quant

    _not_loading(monkeypatch)
    op = quant.api("per_group_quant_fp8@1.0", quant._run_fp8, native="quant_fp8")(quant.per_group_quant_fp8.__wrapped__)
    x = workloads.activations(5, 1024, seed=5, device=DEV)
    with pytest.warns(RuntimeWarning, match="_host"):
        got = op(x)
    assert _same(got, quant.per_group_quant_fp8.general(x)) and op(x.float()) is FallbackReason.OUT_OF_CONTRACT


def _same(a, b):
    if isinstance(a, tuple):
        return isinstance(b, tuple) and len(a) == len(b) and all(_same(x, y) for x, y in zip(a, b))
    if not isinstance(a, torch.Tensor):
        return a is b
    if a.dtype != b.dtype or a.shape != b.shape or a.stride() != b.stride() or a.device != b.device:
        return False
    return torch.equal(a.view(torch.uint8), b.view(torch.uint8))


def _check(name, args, kwargs, served):
    torch.cuda.synchronize()
    got = _lib.host_function(name)(args, kwargs)
    want = NATIVE[name].general(*args, **kwargs)
    torch.cuda.synchronize()
    if served is None:  # served exactly where the general path serves it
        served = not isinstance(want, FallbackReason)
    if served:
        assert got is not None and _same(got, want)
    else:
        assert got is None
    again = NATIVE[name](*args, **kwargs)
    torch.cuda.synchronize()
    assert _same(again, want)
    return want


def _fp8(m, n, k, dtype=FP8):
    x = workloads.activations(m, k, seed=m, device=DEV)
    q, s = aklr_amd.per_group_quant_fp8.general(x)
    b, bs = workloads.blockwise_fp8_weight(n, k, seed=n, device=DEV)
    return x, q.float().to(dtype), s, b.float().to(dtype), bs


@pytest.mark.gpu
@pytest.mark.parametrize("t,h", [(1, 128), (7, 7168), (130, 1536)])
def test_quantizers(t, h):
    say(f"host path quantizers t={t} h={h}")
    x = workloads.activations(t, h, seed=t, device=DEV)
    for name in ("quant_fp8", "quant_mxfp8", "quant_mxfp4"):
        _check(name, (x,), {}, True)
        _check(name, (), {"x": x}, True)
        _check(name, (torch.nn.Parameter(x),), {}, True)
        wide = torch.cat([x, x], 1)
        for bad in (x.float(), x[:, : h - 8], wide[:, :h], x.view(-1)[1:].view(-1), x.t(), x[None], x[:0], x.cpu(), None):
            _check(name, (bad,), {}, None)
    _check("quant_mxfp4", (x, True), {}, True)
    _check("quant_mxfp4", (x,), {"shuffle": False}, True)
    _check("quant_mxfp4", (x, 1), {}, False)
    _check("quant_mxfp4", (x, "yes"), {}, False)


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [(1, 16, 128), (5, 144, 384), (48, 2112, 1024), (333, 3072, 512)])
def test_gemm_fp8(m, n, k):
    say(f"host path gemm fp8 {m}x{n}x{k}")
    x, q, s, b, bs = _fp8(m, n, k)
    kb = k // 128
    km, pre, bias = s.t().contiguous(), layouts.shuffle_weight(b), torch.randn(n, device=DEV)
    rm = km.clone()
    rm.is_row_major = True
    P = {"operand_format": "none:preshuffled"}
    name = "gemm_fp8"
    for args, kw in [((q, b, km, bs), {}), ((q, b, s, bs), {"scale_major_mode": "MN"}),
                     ((q, b, km, bs, (128, 128), "K", True, bias, torch.float16), {"operand_format": "none:none"}),
                     ((q, b, km, bs), {"bias": bias, "out_dtype": torch.bfloat16, "block_size": (128, 128), "out": None}),
                     ((q, pre, s.view(m, kb), bs), P), ((q, pre, rm, bs), P), ((q, b, s.view(m, kb), bs), P),
                     ((q, b), {"b_scale": bs, "a_scale": km})]:
        assert isinstance(_check(name, args, kw, True), torch.Tensor)
    _, q5, _, b5, _ = _fp8(m, n, k, E5M2)
    _check(name, (q5, b5, km, bs), {}, True)
    out = torch.empty((m, n), dtype=torch.bfloat16, device=DEV)
    cut = torch.empty(n * k + 1, dtype=torch.uint8, device=DEV)[1:].view(FP8).view(n, k)
    for args, kw in [((q, b, km, bs), {"out": out}), ((q, b.t().contiguous(), km, bs), {"trans_b": False}),
                     ((q, b, km, bs), {"trans_b": 1}), ((q, b, km, bs), {"block_size": [128, 128]}),
                     ((q, b, km, bs), {"block_size": (64, 128)}), ((q, b, km, bs), {"scale_major_mode": "N"}),
                     ((q, pre, km, bs), {}), ((q, pre, s, bs), {"scale_major_mode": "MN", **P}),
                     ((q, pre, km, bs), {"bias": bias, **P}), ((q5, b5, km, bs), P), ((q, b5, km, bs), {}),
                     ((q, b, km, bs), {"out_dtype": torch.float32}), ((q, b, km, bs), {"operand_format": "x"}),
                     ((q, b, km.double(), bs), {}), ((q, b, km, bs), {"bias": bias[1:]}), ((q, b, km, bs), {"bias": bias.double()}),
                     ((q, cut, km, bs), {}), ((q, b, km, bs.cpu()), {}), ((q, b, km[:, :0], bs), {}), ((q.float(), b, km, bs), {}),
                     ((q, b[: n - 8], km, bs), {}), ((q, b, km, 1.0), {}), ((q[:, :64], b[:, :64], km, bs), {})]:
        _check(name, args, kw, False)
    if m > 1 and kb > 1:
        _check(name, (q, pre, s.view(kb, m).t(), bs), P, False)  # a (1, m)-strided a_scale: served by the general path
        _check(name, (q, b, s.t(), bs), {}, False)

    name = "quant_gemm_fp8"
    wide = torch.cat([x, x], 1)[:, :k]  # a row stride of its own
    for args, kw in [((x, b, bs), {}), ((x, pre, bs), P), ((wide, b, bs), {"bias": bias}),
                     ((x, b, bs, bias, torch.float16), {}), ((x,), {"b": b, "b_scale": bs, "out": None})]:
        assert isinstance(_check(name, args, kw, True), torch.Tensor)
    for args, kw in [((x, b, bs), {"out": out}), ((x, pre, bs), {}), ((x.half(), b, bs), {}), ((x, b5, bs), {}),
                     ((x, b, bs, bias[None]), {}), ((x.t().contiguous().t(), b, bs), {}) if m > 1 else ((x[0], b, bs), {}),
                     ((x, b, bs.t()), {}) if bs.shape[0] != bs.shape[1] else ((x, b, bs.double()), {})]:
        _check(name, args, kw, False)


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [(1, 16, 64), (9, 272, 448), (100, 512, 512)])
def test_gemm_mxfp4(m, n, k):
    say(f"host path gemm mxfp4 {m}x{n}x{k}")
    x = workloads.activations(m, k, seed=m, device=DEV)
    q, s = aklr_amd.dynamic_mxfp4_quant.general(x)
    _, ss = aklr_amd.dynamic_mxfp4_quant.general(x, True)
    b, bs = workloads.mxfp4_weight(n, k, seed=n, device=DEV)
    bias = torch.randn(n, device=DEV)
    pre, bss = layouts.shuffle_weight(b), layouts.shuffle_scale(bs)
    R = {"operand_format": "none:none"}
    name = "gemm_mxfp4"
    u8 = lambda t: t.view(torch.uint8)
    for args, kw in [((q, pre, ss, bss), {}), ((q, b, s, bs), R), ((u8(q), b, u8(s), bs), {"bias": bias, **R}),
                     ((q, pre, ss, bss, 1.0, 0.0, True, bias, torch.float16), {"operand_format": "none:preshuffled"})]:
        assert isinstance(_check(name, args, kw, True), torch.Tensor)
    out = torch.empty((m, n), dtype=torch.bfloat16, device=DEV)
    for args, kw in [((q, b, s, bs), {"out": out, **R}), ((q, pre, ss, bss, 1), {}), ((q, pre, ss, bss, 2.0), {}),
                     ((q, pre, ss, bss), {"beta": 1.0}), ((q, b, s, bs), {}), ((q, pre, ss, bss), {"trans_b": False}),
                     ((q, b, s.float(), bs), R), ((q, b, s, bs), {"out_dtype": torch.float32, **R}),
                     ((q, b, s, bs), {"bias": bias.half(), **R}), ((q.cpu(), b, s, bs), R), ((q, b[:, :-16], s, bs), R)]:
        _check(name, args, kw, False)


@pytest.mark.gpu
def test_streams_modes_and_switches(monkeypatch):
    say("host path streams, modes, switches")
    x = workloads.activations(16, 1024, seed=3, device=DEV)
    want = aklr_amd.per_group_quant_fp8.general(x)
    fn = _lib.host_function("quant_fp8")
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):  # the copy that x comes from is queued on this stream, far behind others
        y = torch.zeros_like(x)
        for _ in range(50):
            torch.mm(torch.ones((512, 512), device=DEV), torch.ones((512, 512), device=DEV))
        y.copy_(x)
        got = fn((y,), {})
    side.synchronize()
    assert _same(got, want)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = fn((y,), {})
    for r in range(3):
        y.copy_(x * (r + 1))
        graph.replay()
        torch.cuda.synchronize()
        assert _same(out, aklr_amd.per_group_quant_fp8.general(y))
        torch.cuda.synchronize()
    with torch.device("cpu"):
        assert fn((x,), {}) is None  # a function mode is active
    monkeypatch.setenv("AKLR_DISABLE", "per_group_quant_fp8@1.0")
    assert fn((x,), {}) is None and aklr_amd.per_group_quant_fp8(x) is FallbackReason.DISABLED
    monkeypatch.setenv("AKLR_DISABLE", "0")
    assert fn((x,), {}) is not None
    monkeypatch.setenv("AKLR_TRACE", "op")
    assert fn((x,), {}) is None
    monkeypatch.setenv("AKLR_TRACE", "loud")
    with pytest.raises(ValueError):
        aklr_amd.per_group_quant_fp8(x)
    monkeypatch.delenv("AKLR_TRACE")
    torch.use_deterministic_algorithms(True)
    try:
        assert fn((x,), {}) is None
    finally:
        torch.use_deterministic_algorithms(False)

    class Sub(torch.Tensor):
        pass

    assert fn((x.as_subclass(Sub),), {}) is None
