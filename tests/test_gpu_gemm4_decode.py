"""The MXFP4 decode plans of preshuffled weights (m <= 16) at the edges of their rule: 224, 304, 512, 768, 1024,
1536 and 1792 column tiles, 240 workgroups of 224 columns, 132 groups of 32, K around 4096, 7936, 8192 and 16384,
K that ends inside a 256-value block, one row and sixteen.

Against the products in float64: the operands' products are exact in fp32, so an output is off by at most
the fp32 sum of k terms, k * 2^-24 * sum |a||b|, and its one rounding to bf16, 2^-8 |y|."""
from __future__ import annotations

import pytest
import torch

import aklr_amd
from aklr_amd import _lib, layouts, workloads
from tests.helpers import say

DEV = "cuda:0"
PRE = (_lib.B_PRESHUFFLE_16x16, _lib.SCALES_SHUFFLED)


@pytest.mark.parametrize("m,n,k,kernel", [
    (1, 3568, 8192, 0), (1, 3584, 8192, 1), (16, 28672, 8192, 1), (1, 28688, 8192, 0), (16, 28688, 4096, 0),
    (8, 57344, 8192, 0), (9, 57344, 4032, 0), (8, 10240, 8256, 0), (8, 8192, 28672, 0), (17, 4096, 4096, 1),
    (33, 4096, 4096, 2), (1, 4864, 8192, 1), (16, 4880, 8192, 0), (16, 4880, 7936, 1), (1, 8192, 8192, 1),
    (7, 8208, 8192, 0), (8, 8208, 8192, 1), (1, 12288, 4096, 1), (11, 12304, 4096, 0), (12, 12304, 4096, 1),
    (16, 12304, 4032, 0), (16, 16384, 8192, 1), (16, 16400, 8192, 0), (16, 24576, 8192, 0), (16, 24592, 8192, 1),
    (11, 57344, 8192, 0), (12, 57344, 8192, 1), (16, 57360, 8192, 0), (16, 53536, 8192, 0), (16, 53552, 8192, 1),
])
def test_which_kernel(native_lib, m, n, k, kernel):
    assert native_lib.aklr_gemm_a4w4_mxfp4_kernel(m, n, k, *PRE) == kernel
    if m <= 16:
        assert native_lib.aklr_gemm_a4w4_mxfp4_kernel(m, n, k, _lib.B_ROW_MAJOR, _lib.SCALES_ROW_MAJOR) == 0


def _dequantized(codes, scales):
    lut = torch.tensor([0, 0.5, 1, 1.5, 2, 3, 4, 6, 0, -0.5, -1, -1.5, -2, -3, -4, -6], dtype=torch.float64, device=DEV)
    c = codes.view(torch.uint8)
    v = torch.stack((lut[(c & 15).long()], lut[(c >> 4).long()]), -1).view(c.shape[0], -1)
    return v * torch.exp2(scales.view(torch.uint8).double() - 127).repeat_interleave(32, 1)


@pytest.mark.gpu
@pytest.mark.parametrize("m", [1, 5, 16])
@pytest.mark.parametrize("n,k", [(3568, 512), (3584, 64), (3584, 448), (4096, 8192), (10240, 2048), (10256, 320),
                                 (24576, 1536), (28672, 576), (28688, 4096), (3584, 16448), (4096, 16640),
                                 (4128, 17408), (12304, 4160), (28672, 4096), (53776, 4096), (4224, 18496)])
def test_decode_plans(m, n, k):
    say(f"mxfp4 decode m={m} n={n} k={k}")
    x = workloads.activations(m, k, seed=m + n, device=DEV)
    a, sa = aklr_amd.dynamic_mxfp4_quant(x, shuffle=False)
    b, sb = workloads.mxfp4_weight(n, k, seed=k, device=DEV)
    bias = torch.randn(n, device=DEV)
    a_s = aklr_amd.dynamic_mxfp4_quant(x, shuffle=True)[1]
    bp, sbp = layouts.shuffle_weight(b), layouts.shuffle_scale(sb)
    out = aklr_amd.gemm_a4w4_mxfp4(a, bp, a_s, sbp, bias=bias)
    half = aklr_amd.gemm_a4w4_mxfp4(a, bp, a_s, sbp, out_dtype=torch.float16)
    again = aklr_amd.gemm_a4w4_mxfp4(a, bp, a_s, sbp, bias=bias)
    torch.cuda.synchronize()
    da, db = _dequantized(a, sa), _dequantized(b, sb)
    y, total = da @ db.t(), da.abs() @ db.abs().t()
    for got, ref, eps in ((out, y + bias.double(), 2.0**-8), (half, y, 2.0**-11)):
        bound = (k + 2) * 2.0**-24 * (total + bias.abs().double()) + eps * ref.abs() + 2.0**-24
        assert bool(((got.double() - ref).abs() <= bound).all())
    assert torch.equal(out.view(torch.int16), again.view(torch.int16))
