"""GPU checks of the launches around the grouped MoE GEMMs at the edges of their plans: the router's three
tile shapes and its K ranges, the grouped top-k at one and four scores a lane batch (up to 256 and up to
1024 experts), the expert sort past one batch of ids, and the combine past one batch of slots.

- Router and top-k: inputs are small dyadic values, so logits are exact in fp32 in every order; the whole
  op must then equal, bit for bit, ``moe_fp8_route`` on those logits (rounded to bf16 by torch) followed by
  ``moe_fp8_experts``. The picks are checked against the oracle's grouped top-k, near-ties aside (two
  sigmoids within 1e-6 relative).
- Combine: slots past the ninth against the same call with the slots of one token spread over tokens of
  its own, summed in float64: each of the S terms is rounded to bf16 once (2^-9 relative) and so is the
  sum, so |diff| <= 2^-8 (sum of |terms| + |result|).
"""
from __future__ import annotations

import numpy as np
import pytest
import torch

import aklr_amd
from oracle import moe
from tests.helpers import f32, say
from tests.test_gpu_moe import _routing_tie

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _weights(e, d, inter, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    w1 = (torch.randn((e, 2 * inter, d), device=DEV, generator=g) * 64).to(torch.float8_e4m3fn)
    w2 = (torch.randn((e, d, inter), device=DEV, generator=g) * 64).to(torch.float8_e4m3fn)
    s1 = torch.rand((e, 2 * inter // 128, d // 128), device=DEV, generator=g) / 512 + 2**-12
    s2 = torch.rand((e, d // 128, inter // 128), device=DEV, generator=g) / 512 + 2**-12
    return w1, s1, w2, s2


# tile edges (16, 32 and 64 tokens; 16, 32 and 256 experts), one K range and sixteen, fewer K steps than waves
@pytest.mark.parametrize("t,e,g,tg,d", [
    (1, 16, 1, 1, 128), (15, 40, 8, 4, 256), (16, 256, 8, 4, 7168), (17, 258, 1, 1, 384), (33, 1024, 8, 4, 1024),
    (130, 65, 1, 1, 2048), (1023, 64, 8, 4, 128), (1024, 320, 8, 4, 256), (1089, 256, 1, 1, 896), (1500, 32, 8, 4, 512),
])
def test_whole_op_equals_route_and_experts(t, e, g, tg, d):
    say(f"moe router t={t} e={e} groups={g}/{tg} d={d}")
    inter, topk = 128, 8
    gen = torch.Generator(device=DEV).manual_seed(t + e)
    x = (torch.randint(-8, 9, (t, d), device=DEV, generator=gen) / 8).to(torch.bfloat16)
    r = (torch.randint(-8, 9, (e, d), device=DEV, generator=gen) / 64).to(torch.bfloat16)
    bias = (torch.randn(e, device=DEV, generator=gen) * 0.05).to(torch.bfloat16)
    w1, s1, w2, s2 = _weights(e + 1, d, inter, t)
    out = aklr_amd.deepseek_v2_fp8_moe(x, r, bias, w1, s1, w2, s2, topk, g, tg, True, "sigmoid", 2.5)
    logits = (x.double() @ r.double().t()).to(torch.bfloat16)
    ids, weights = aklr_amd.moe_fp8_route(logits, bias, topk, g, tg, True, 2.5)
    want = aklr_amd.moe_fp8_experts(x, w1, w2, weights, ids, s1, s2)
    torch.cuda.synchronize()
    assert torch.equal(out.view(torch.int16), want.view(torch.int16))

    lg, bs = f32(logits), f32(bias)
    ids_o, w_o = moe.grouped_topk(lg, bs, topk, g, tg, True, 2.5)
    biased = (moe.sigmoid32(lg) + bs).astype(np.float32)
    got, got_w = ids.cpu().numpy(), weights.cpu().numpy()
    ties = 0
    for i in range(t):
        if np.array_equal(got[i, :topk], ids_o[i]):
            np.testing.assert_allclose(got_w[i, :topk], w_o[i], rtol=1e-5)
        else:
            close = np.allclose(biased[i][got[i, :topk]], biased[i][ids_o[i]], rtol=1e-6, atol=0)
            assert close or _routing_tie(biased[i], topk, g, tg), f"token {i}"
            ties += 1
    assert ties <= max(1, 0.05 * t)


@pytest.mark.parametrize("e,g,tg", [(64, 1, 1), (256, 8, 4), (512, 8, 4)])
def test_route_skips_nan_and_orders_infinities(e, g, tg):
    say(f"moe route special values e={e}")
    gen = torch.Generator().manual_seed(e)
    lg = torch.randn((6, e), generator=gen).to(torch.bfloat16).float()
    lg[1, 3] = float("nan")       # never picked
    lg[2, e - 1] = float("inf")   # score 1: first
    lg[3, : e - 9] = float("-inf")  # score 0: picked only by their bias
    bias = (torch.rand(e, generator=gen) * 0.01).to(torch.bfloat16)
    ids, _ = aklr_amd.moe_fp8_route(lg.to(torch.bfloat16).to(DEV), bias.to(DEV), 8, g, tg, True, 1.0, append_shared=False)
    got = ids.cpu().numpy()
    lg_o = lg.numpy().copy()
    bias_rows = np.repeat(bias.float().numpy()[None], 6, 0)
    lg_o[1, 3], bias_rows[1, 3] = 0.0, -np.inf
    for i in range(6):
        want, _ = moe.grouped_topk(lg_o[i : i + 1], bias_rows[i], 8, g, tg, True, 1.0)
        biased = (moe.sigmoid32(lg_o[i]) + bias_rows[i]).astype(np.float32)
        assert np.array_equal(got[i], want[0]) or np.allclose(biased[got[i]], biased[want[0]], rtol=1e-6, atol=0), i
    assert 3 not in got[1]


@pytest.mark.parametrize("slots,d", [(1, 128), (9, 1024), (10, 1152), (19, 2176), (63, 256)])
def test_combine_slot_batches(slots, d):
    say(f"moe combine slots={slots} d={d}")
    e, inter, t = 7, 128, 5
    gen = torch.Generator(device=DEV).manual_seed(slots)
    x = torch.randn((t, d), device=DEV, generator=gen).to(torch.bfloat16)
    ids = torch.randint(-1, e + 1, (t, slots), device=DEV, generator=gen).to(torch.int32)  # -1 and e: skipped
    wts = torch.rand((t, slots), device=DEV, generator=gen) + 0.1
    w1, s1, w2, s2 = _weights(e, d, inter, slots)
    out = aklr_amd.moe_fp8_experts(x, w1, w2, wts, ids, s1, s2)
    one = aklr_amd.moe_fp8_experts(x.repeat_interleave(slots, 0).contiguous(), w1, w2,
                                   torch.ones((t * slots, 1), device=DEV), ids.reshape(-1, 1).contiguous(), s1, s2)
    torch.cuda.synchronize()
    terms = one.double().view(t, slots, d) * wts.double()[..., None]
    want = terms.sum(1)
    bound = 2.0**-8 * (terms.abs().sum(1) + want.abs()) + 1e-30
    assert bool(((out.double() - want).abs() <= bound).all())
