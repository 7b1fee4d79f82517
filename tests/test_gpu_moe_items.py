"""The grouped down GEMM's items of several weight tiles: where the blocks times the weight tiles leave four
items a CU, an item takes up to 16 K steps' worth of tiles. Every token's result depends on that token
alone and is summed in the same order in every block class, so a call whose items hold several tiles must
equal, bit for bit, calls on a few of its tokens at a time, whose items hold one (their blocks are too few).
Sizes: one to three K blocks, a last item with fewer tiles, a last tile with 128 of its 256 columns, all
three block classes."""
from __future__ import annotations

import pytest
import torch

import aklr_amd
from aklr_amd import layouts
from tests.helpers import say

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("e,d,inter,t,shuffled", [(257, 7168, 128, 120, True), (257, 7168, 256, 120, False),
                                                  (900, 1152, 128, 420, True), (500, 2176, 384, 260, False)])
def test_items_of_several_tiles(e, d, inter, t, shuffled):
    say(f"moe items e={e} d={d} inter={inter} t={t}")
    g = torch.Generator(device=DEV).manual_seed(e + d)
    w1 = (torch.randn((e, 2 * inter, d), device=DEV, generator=g) * 64).to(torch.float8_e4m3fn)
    w2 = (torch.randn((e, d, inter), device=DEV, generator=g) * 64).to(torch.float8_e4m3fn)
    s1 = torch.rand((e, 2 * inter // 128, d // 128), device=DEV, generator=g) / 512 + 2**-12
    s2 = torch.rand((e, d // 128, inter // 128), device=DEV, generator=g) / 512 + 2**-12
    if shuffled:
        w1, w2 = layouts.shuffle_weight(w1), layouts.shuffle_weight(w2)
    x = torch.randn((t, d), device=DEV, generator=g).to(torch.bfloat16)
    ids = torch.randint(0, e, (t, 9), device=DEV, generator=g).to(torch.int32)
    ids[:, 0] = 3                       # a 256-row block where t > 128
    ids[: min(t, 100), 1] = 5           # a 128-row block
    wts = torch.rand((t, 9), device=DEV, generator=g)
    tiles = -(-d // 256)
    assert torch.unique(ids).numel() * tiles >= 2 * 4 * 256, "items of two tiles or more"
    out = aklr_amd.moe_fp8_experts(x, w1, w2, wts, ids, s1, s2)
    step = max(1, 2 * 4 * 256 // (tiles * 9) - 1)
    parts = [aklr_amd.moe_fp8_experts(x[i : i + step].contiguous(), w1, w2, wts[i : i + step].contiguous(),
                                      ids[i : i + step].contiguous(), s1, s2) for i in range(0, t, step)]
    torch.cuda.synchronize()
    assert torch.equal(out.view(torch.int16), torch.cat(parts).view(torch.int16))


@pytest.mark.parametrize("value", [float("inf"), float("nan")])
@pytest.mark.parametrize("e,d,inter,t,shuffled", [(257, 7168, 256, 120, True), (900, 1152, 128, 420, False)])
def test_a_scale_that_is_not_finite_stays_in_its_columns(e, d, inter, t, shuffled, value):
    """Every second weight tile's scales of the last K block are not finite, in every expert: the columns of
    the other tiles must equal a clean call's bit for bit, the tiles before them in an item or not."""
    say(f"moe items, scales of {value} e={e} d={d} inter={inter} t={t}")
    g = torch.Generator(device=DEV).manual_seed(e + d)
    w1 = (torch.randn((e, 2 * inter, d), device=DEV, generator=g) * 64).to(torch.float8_e4m3fn)
    w2 = (torch.randn((e, d, inter), device=DEV, generator=g) * 64).to(torch.float8_e4m3fn)
    s1 = torch.rand((e, 2 * inter // 128, d // 128), device=DEV, generator=g) / 512 + 2**-12
    s2 = torch.rand((e, d // 128, inter // 128), device=DEV, generator=g) / 512 + 2**-12
    if shuffled:
        w1, w2 = layouts.shuffle_weight(w1), layouts.shuffle_weight(w2)
    x = torch.randn((t, d), device=DEV, generator=g).to(torch.bfloat16)
    ids = torch.randint(0, e, (t, 9), device=DEV, generator=g).to(torch.int32)
    ids[: min(t, 100), 1] = 5           # a 128-row block
    wts = torch.rand((t, 9), device=DEV, generator=g)
    assert torch.unique(ids).numel() * -(-d // 256) >= 2 * 4 * 256, "items of two tiles or more"
    bad = s2.clone()
    hit = (torch.arange(d // 128, device=DEV) // 2) % 2 == 0
    bad[:, hit, -1] = value
    clean = aklr_amd.moe_fp8_experts(x, w1, w2, wts, ids, s1, s2)
    out = aklr_amd.moe_fp8_experts(x, w1, w2, wts, ids, s1, bad)
    torch.cuda.synchronize()
    cols = hit.repeat_interleave(128)
    assert torch.equal(out[:, ~cols].view(torch.int16), clean[:, ~cols].view(torch.int16))
    assert not bool(torch.isfinite(out[:, cols]).any())
