"""The MXFP4 LDS kernel's 256-row tiles of preshuffled weights, whose K loop has two barriers a step from
K = 4096 on and one below: both tile widths, one K step, step counts around 16 (the loop's slots turn every 2,
3 or 4 steps), rows and columns that end inside a tile, bias, both output types, both scale layouts.

Against the products in float64: the operands' products are exact in fp32, so an output is off by at most
the fp32 sum of k terms, k * 2^-24 * sum |a||b|, and its one rounding to the output type."""
from __future__ import annotations

import ctypes

import pytest
import torch

import aklr_amd
from aklr_amd import _lib, layouts, workloads
from tests.helpers import say

DEV = "cuda:0"
PRE = _lib.B_PRESHUFFLE_16x16


def _tile(lib, m, n, k, layout):
    v = [ctypes.c_int(-1) for _ in range(3)]
    got = lib.aklr_gemm_a4w4_mxfp4_tile(m, n, k, layout, *(ctypes.byref(x) for x in v))
    return tuple(x.value for x in v) if got else None


def test_which_tile(native_lib):
    assert _tile(native_lib, 1000, 10256, 4096, PRE) == (256, 256, 2)
    assert _tile(native_lib, 1000, 10256, 3840, PRE) == (256, 256, 1)
    assert _tile(native_lib, 1000, 10256, 4096, _lib.B_ROW_MAJOR) == (256, 256, 1)
    assert _tile(native_lib, 300, 272, 4096, PRE) == (128, 128, 1)
    assert _tile(native_lib, 32, 10256, 4096, PRE) is None and _tile(native_lib, 1000, 10256, 4160, PRE) is None


def _dequantized(codes, scales):
    lut = torch.tensor([0, 0.5, 1, 1.5, 2, 3, 4, 6, 0, -0.5, -1, -1.5, -2, -3, -4, -6], dtype=torch.float64, device=DEV)
    c = codes.view(torch.uint8)
    v = torch.stack((lut[(c & 15).long()], lut[(c >> 4).long()]), -1).view(c.shape[0], -1)
    return v * torch.exp2(scales.view(torch.uint8).double() - 127).repeat_interleave(32, 1)


@pytest.mark.gpu
@pytest.mark.parametrize("k", [256, 768, 3840, 4096, 4352, 4608, 4864])
@pytest.mark.parametrize("m,n,cols", [(389, 16480, 256), (135, 16720, 128), (700, 8208, 128)])
def test_tiles(native_lib, m, n, cols, k):
    say(f"mxfp4 tiles m={m} n={n} k={k}")
    assert _tile(native_lib, m, n, k, PRE) == (256, cols, 2 if k >= 4096 else 1)
    x = workloads.activations(m, k, seed=m + n, device=DEV)
    a, sa = aklr_amd.dynamic_mxfp4_quant(x, shuffle=False)
    b, sb = workloads.mxfp4_weight(n, k, seed=k, device=DEV)
    bias = torch.randn(n, device=DEV)
    a_s = aklr_amd.dynamic_mxfp4_quant(x, shuffle=True)[1]
    bp, sbp = layouts.shuffle_weight(b), layouts.shuffle_scale(sb)
    out = aklr_amd.gemm_a4w4_mxfp4(a, bp, a_s, sbp, bias=bias)
    half = aklr_amd.gemm_a4w4_mxfp4(a, bp, a_s, sbp, out_dtype=torch.float16)
    # preshuffled weights with row-major scales: the C ABI takes them, the op does not
    rows = torch.empty_like(out)
    u8 = lambda t: t.view(torch.uint8)
    ws = torch.empty(max(16, native_lib.aklr_gemm_a4w4_mxfp4_workspace_bytes(m, n, k)), dtype=torch.uint8, device=DEV)
    _lib.check(native_lib.aklr_gemm_a4w4_mxfp4(
        u8(a).data_ptr(), k // 2, u8(bp).data_ptr(), k // 2, u8(sa).data_ptr(), k // 32, u8(sb).data_ptr(), k // 32,
        bias.data_ptr(), rows.data_ptr(), n, m, n, k, PRE, _lib.SCALES_ROW_MAJOR, _lib.OUT_BF16, ws.data_ptr(),
        ws.numel(), torch.cuda.current_stream().cuda_stream), "row-major scales")
    torch.cuda.synchronize()
    da, db = _dequantized(a, sa), _dequantized(b, sb)
    y, total = da @ db.t(), da.abs() @ db.abs().t()
    for got, ref, eps in ((out, y + bias.double(), 2.0**-8), (half, y, 2.0**-11)):
        bound = (k + 2) * 2.0**-24 * (total + bias.abs().double()) + eps * ref.abs() + 2.0**-24
        assert bool(((got.double() - ref).abs() <= bound).all())
    assert torch.equal(rows.view(torch.int16), out.view(torch.int16))
