"""The work that a user of this library has it do, as cases that can be timed and compared.

A serving program calls these ops for every layer of every step, so the cases are its single layers, each
through the public entry points, from the smallest decode call to a full prefill:

- ``quant_fp8`` / ``quant_mxfp8``: an activation quantizer on its own;
- ``linear_fp8``: an FP8 linear layer, ``per_group_quant_fp8`` then ``gemm_a8w8_blockwise_scaled``;
- ``fused_fp8``: the same layer as one ``quant_gemm_a8w8_blockwise_scaled`` call;
- ``gemm_fp8``: the FP8 GEMM on activations that are quantized already;
- ``linear_mxfp4``: an MXFP4 linear layer, ``dynamic_mxfp4_quant`` then ``gemm_a4w4_mxfp4``;
- ``moe_layer``: a whole mixture-of-experts layer, ``deepseek_v2_fp8_moe``;
- ``moe_experts``: its two halves on given router logits, ``moe_fp8_route`` then ``moe_fp8_experts``.

Values: activations N(0, 1) with 1% outliers of 20 times that; weights N(0, 0.02), quantized per 128 x 128
block (FP8) or per 32 values (MXFP4).
"""
from __future__ import annotations

import torch

import aklr_amd
from aklr_amd import layouts, workloads

DEV = "cuda:0"
F64 = torch.float64
TOPK = 8
OUT = {"bf16": torch.bfloat16, "f16": torch.float16}

# (N, K) of the FP8 linears: the decode / prefill configurations' layers, a tensor-parallel shard of one,
# and the square and narrow layers the benchmark also times
FP8_NK = ((2112, 7168), (24576, 1536), (7168, 16384), (3072, 1536), (7168, 2048), (4096, 4096), (4096, 8192),
          (512, 4096), (1536, 4096), (8192, 1024), (32768, 1024), (4096, 512))
MXFP4_NK = ((10240, 8192), (57344, 8192), (8192, 28672), (8192, 8192), (4096, 4096), (7168, 2048))


def listed():
    return [
        # a decode batch's activations on their way into an FP8 linear: the smallest call there is
        {"name": "quant_fp8_decode", "op": "quant_fp8", "m": 8, "k": 7168},
        # the latent down-projection of one decoding sequence, quantization fused: latency alone
        {"name": "fused_fp8_m1", "op": "fused_fp8", "m": 1, "n": 2112, "k": 7168, "layout": "shuffled"},
        # the attention output projection of a decode batch: a long stream of weights (the headline shape)
        {"name": "linear_fp8_m16", "op": "linear_fp8", "m": 16, "n": 7168, "k": 16384, "layout": "shuffled"},
        # the query up-projection of a large decode batch
        {"name": "linear_fp8_m128", "op": "linear_fp8", "m": 128, "n": 24576, "k": 1536, "layout": "shuffled"},
        # a ragged chunk of prefill through one tensor-parallel shard, weights as the checkpoint has them,
        # K-major scales, with a bias and fp16 results
        {"name": "gemm_fp8_ragged", "op": "gemm_fp8", "m": 333, "n": 3072, "k": 1536, "layout": "row_major",
         "bias": True, "out": "f16"},
        # a full prefill through the largest FP8 linear
        {"name": "linear_fp8_m4096", "op": "linear_fp8", "m": 4096, "n": 7168, "k": 16384, "layout": "shuffled"},
        # the fused query/key/value projection of a small decode batch in MXFP4
        {"name": "linear_mxfp4_m8", "op": "linear_mxfp4", "m": 8, "n": 10240, "k": 8192, "layout": "shuffled"},
        # the same layer at prefill
        {"name": "linear_mxfp4_m4096", "op": "linear_mxfp4", "m": 4096, "n": 10240, "k": 8192, "layout": "shuffled"},
        # a prefill's activations in MXFP8, an odd number of tokens
        {"name": "quant_mxfp8_prefill", "op": "quant_mxfp8", "m": 5003, "k": 7168},
        # a mixture-of-experts layer of a few decoding sequences: a few experts' weights and seven launches
        {"name": "moe_layer_t4", "op": "moe_layer", "m": 4, "e": 256, "d": 7168, "i": 2048, "layout": "shuffled"},
        # the same layer of a decode batch on one of eight tensor-parallel ranks (each expert cut to 256)
        {"name": "moe_layer_tp8_t128", "op": "moe_layer", "m": 128, "e": 256, "d": 7168, "i": 256,
         "layout": "shuffled"},
        # the experts of a full prefill on a skewed routing: a few experts with many rows, many with few
        {"name": "moe_experts_t4096", "op": "moe_experts", "m": 4096, "e": 256, "d": 7168, "i": 2048,
         "layout": "shuffled"},
    ]


def _log_uniform(rng, lo, hi):
    return min(hi, max(lo, int(round(lo * (hi / lo) ** rng.random()))))


def draw(rng):
    op = rng.choice(("quant_fp8", "fused_fp8", "linear_fp8", "linear_fp8", "linear_fp8", "gemm_fp8", "linear_mxfp4",
                     "linear_mxfp4", "quant_mxfp8", "moe_layer", "moe_layer", "moe_experts"))
    case = {"op": op}
    if op in ("quant_fp8", "quant_mxfp8"):
        case.update(m=_log_uniform(rng, 1, 16384), k=rng.choice((1536, 2048, 4096, 7168, 16384)))
    elif op in ("linear_fp8", "gemm_fp8", "fused_fp8"):
        n, k = rng.choice(FP8_NK)
        case.update(m=_log_uniform(rng, 1, 16 if op == "fused_fp8" else 8192), n=n, k=k)
        case["layout"] = "row_major" if op == "gemm_fp8" else rng.choice(("shuffled", "shuffled", "row_major"))
        if op == "gemm_fp8":
            case.update(bias=rng.random() < 0.5, out=rng.choice(("bf16", "f16")))
    elif op == "linear_mxfp4":
        n, k = rng.choice(MXFP4_NK)
        case.update(m=_log_uniform(rng, 1, 4096), n=n, k=k, layout=rng.choice(("shuffled", "shuffled", "row_major")))
    else:
        # experts whole, or cut for 2, 4 or 8 tensor-parallel ranks; layers of 32 to 256 routed experts
        case.update(m=_log_uniform(rng, 1, 4000), e=rng.choice((32, 64, 128, 256)), d=7168,
                    i=rng.choice((256, 512, 1024, 2048)), layout=rng.choice(("shuffled", "shuffled", "row_major")))
    return case


# ---------------------------------------------------------------------------------------------
# inputs
def _seed(seed, salt):
    return seed * 4099 + salt  # an expert stack draws one seed per expert, so states lie further apart than that


def _generator(seed, salt):
    return workloads.generator(_seed(seed, salt), DEV)


def _activations(case, seed):
    return workloads.activations(case["m"], case.get("k", case.get("d")), seed=_seed(seed, 4000), device=DEV)


def _fp8_weight(case, seed):
    return workloads.blockwise_fp8_weight(case["n"], case["k"], seed=_seed(seed, 4001), device=DEV)


def _mxfp4_weight(case, seed):
    """Quantized in row blocks, so that the largest layer's temporaries stay small."""
    g = _generator(seed, 4002)
    codes, scales = [], []
    for r in range(0, case["n"], 8192):
        w = torch.randn((min(8192, case["n"] - r), case["k"]), generator=g, device=DEV) * 0.02
        c, s = workloads.mxfp4_quantize(w)
        codes.append(c)
        scales.append(s)
    return torch.cat(codes), torch.cat(scales)


def _bias(case, seed):
    return torch.randn(case["n"], generator=_generator(seed, 4003), device=DEV) * 0.5 if case.get("bias") else None


def _experts(case, seed):
    w1, s1 = workloads.moe_expert_weights(case["e"] + 1, 2 * case["i"], case["d"], seed=_seed(seed, 0), device=DEV)
    w2, s2 = workloads.moe_expert_weights(case["e"] + 1, case["d"], case["i"], seed=_seed(seed, 1500), device=DEV)
    return w1, s1, w2, s2


def _router(case, seed):
    """(hidden, router weight, correction bias). Hidden states and router weights lie on the grids 2^-5 and
    2^-9, which their magnitudes (up to 4 and 0.1) keep within bf16's 8 bits or round to: every product and
    every partial sum of a logit is then exact in fp32, whatever the order, so that one routing is right and
    a sum in another order does not send a token to another expert."""
    g = _generator(seed, 4004)
    x = torch.randn((case["m"], case["d"]), generator=g, device=DEV).clamp(-3.9, 3.9)
    x = (torch.round(x * 32) / 32).to(torch.bfloat16)
    w = torch.randn((case["e"], case["d"]), generator=g, device=DEV) * 0.02
    w = (torch.round(w * 512) / 512).to(torch.bfloat16)
    bias = (torch.randn(case["e"], generator=g, device=DEV) * 0.05).to(torch.bfloat16)
    return x, w, bias


def _logits(case, seed):
    """Router logits whose eight best follow Zipf(1.1) over the experts (log-probabilities plus Gumbel
    noise): the skew of a served batch."""
    g = _generator(seed, 4005)
    p = torch.arange(1, case["e"] + 1, device=DEV, dtype=torch.float32).pow(-1.1)
    u = torch.rand((case["m"], case["e"]), generator=g, device=DEV).clamp(1e-7, 1 - 1e-7)
    logits = torch.log(p / p.sum()) - torch.log(-torch.log(u))
    return logits.to(torch.bfloat16), torch.zeros(case["e"], dtype=torch.bfloat16, device=DEV)


def _shuffle(case, w):
    return layouts.shuffle_weight(w) if case["layout"] == "shuffled" else w


def _format(case):
    return "none:preshuffled" if case["layout"] == "shuffled" else "none:none"


def prepare(case, seed):
    op = case["op"]
    state = {"case": dict(case)}
    if op in ("quant_fp8", "quant_mxfp8"):
        state["x"] = _activations(case, seed)
    elif op in ("linear_fp8", "fused_fp8", "gemm_fp8"):
        x = _activations(case, seed)
        b, state["b_scale"] = _fp8_weight(case, seed)
        state["b"] = _shuffle(case, b)
        state["bias"] = _bias(case, seed)
        if op == "gemm_fp8":
            q, s = aklr_amd.per_group_quant_fp8(x)
            state["q"], state["a_scale"] = q, s.t().contiguous()
        else:
            state["x"] = x
    elif op == "linear_mxfp4":
        state["x"] = _activations(case, seed)
        b, s = _mxfp4_weight(case, seed)
        state["b"] = _shuffle(case, b)
        state["b_scale"] = layouts.shuffle_scale(s) if case["layout"] == "shuffled" else s
    else:
        w1, state["s1"], w2, state["s2"] = _experts(case, seed)
        state["w1"], state["w2"] = _shuffle(case, w1), _shuffle(case, w2)
        if op == "moe_layer":
            state["x"], state["router"], state["correction"] = _router(case, seed)
        else:
            state["x"] = _activations(case, seed)
            state["logits"], state["correction"] = _logits(case, seed)
    return state


# ---------------------------------------------------------------------------------------------
# one pass
def run(state):
    case = state["case"]
    op = case["op"]
    if op == "quant_fp8":
        return aklr_amd.per_group_quant_fp8(state["x"])
    if op == "quant_mxfp8":
        return aklr_amd.per_group_quant_mxfp8(state["x"])
    if op == "fused_fp8":
        return aklr_amd.quant_gemm_a8w8_blockwise_scaled(state["x"], state["b"], state["b_scale"],
                                                         operand_format=_format(case))
    if op == "linear_fp8":
        q, s = aklr_amd.per_group_quant_fp8(state["x"])
        if case["layout"] == "shuffled":  # the quantizer's scales are the column-major ones this layout takes
            return aklr_amd.gemm_a8w8_blockwise_scaled(q, state["b"], s.view(case["m"], case["k"] // 128),
                                                       state["b_scale"], operand_format="none:preshuffled")
        return aklr_amd.gemm_a8w8_blockwise_scaled(q, state["b"], s, state["b_scale"], scale_major_mode="MN")
    if op == "gemm_fp8":
        return aklr_amd.gemm_a8w8_blockwise_scaled(state["q"], state["b"], state["a_scale"], state["b_scale"],
                                                   bias=state["bias"], out_dtype=OUT[case["out"]])
    if op == "linear_mxfp4":
        q, s = aklr_amd.dynamic_mxfp4_quant(state["x"], shuffle=case["layout"] == "shuffled")
        return aklr_amd.gemm_a4w4_mxfp4(q, state["b"], s, state["b_scale"], operand_format=_format(case))
    if op == "moe_layer":
        return aklr_amd.deepseek_v2_fp8_moe(state["x"], state["router"], state["correction"], state["w1"], state["s1"],
                                            state["w2"], state["s2"], TOPK, 8, 4, True, "sigmoid", 2.5)
    ids, weights = aklr_amd.moe_fp8_route(state["logits"], state["correction"], TOPK, 1, 1, True, 2.5)
    out = aklr_amd.moe_fp8_experts(state["x"], state["w1"], state["w2"], weights, ids, state["s1"], state["s2"])
    return {"ids": ids, "weights": weights, "out": out}


# ---------------------------------------------------------------------------------------------
# what a pass cannot do without
def _touched(case):
    """The experts a routing is expected to reach, the shared one among them."""
    m, e = case["m"], case["e"]
    if case["op"] == "moe_layer":
        return 1 + e * (1 - (1 - TOPK / e) ** m)
    p = [(j + 1) ** -1.1 for j in range(e)]
    total = sum(p)
    return 1 + sum(1 - (1 - v / total) ** (TOPK * m) for v in p)


def work(case):
    op, m = case["op"], case["m"]
    if op in ("quant_fp8", "quant_mxfp8"):
        return {"bytes": 3 * m * case["k"] + m * case["k"] // 32, "flops": 0}  # 4 bytes per 128 values, or 1 per 32
    if op in ("linear_fp8", "fused_fp8", "gemm_fp8"):
        n, k = case["n"], case["k"]
        a = m * k + 4 * m * k // 128 if op == "gemm_fp8" else 2 * m * k
        return {"bytes": a + n * k + 4 * -(-n // 128) * k // 128 + (4 * n if case.get("bias") else 0) + 2 * m * n,
                "flops": 2 * m * n * k}
    if op == "linear_mxfp4":
        n, k = case["n"], case["k"]
        return {"bytes": 2 * m * k + n * k // 2 + n * k // 32 + 2 * m * n, "flops": 2 * m * n * k}
    e, d, i = case["e"], case["d"], case["i"]
    weights = _touched(case) * 3 * d * i * (1 + 4 / 128 ** 2)
    router = 2 * e * (d + 1) if op == "moe_layer" else 2 * e * (m + 1) + 8 * m * (TOPK + 1)
    return {"bytes": weights + router + 4 * m * d,
            "flops": 2 * m * (TOPK + 1) * 3 * d * i + (2 * m * e * d if op == "moe_layer" else 0)}


def tolerance(case):
    op = case["op"]
    if op in ("quant_fp8", "quant_mxfp8"):
        return "exact"  # the formula fixes every rounding, so codes and scales are the same bits
    if op == "moe_layer":
        return {"rel": 1.2e-2}
    if op == "moe_experts":
        # the picks are whole values: a near-tie of two sigmoids may go either way
        return {"rel": 1.2e-2, "differ": 1e-3}
    # fp32 sums of exact products, rounded once to bf16 or fp16
    return {"rel": 1e-3 if case.get("out") == "f16" else 7e-3}


# ---------------------------------------------------------------------------------------------
# the same in 64 bits, in plain torch
def _groups_fp8(x, divide):
    """The FP8 quantizer's codes and scales per 128 values, in the fp32 steps that define it: as a decoded
    fp32 tensor and the scales [rows, K/128]. ``divide``: the mixture-of-experts layers' scale, amax / 448."""
    x = x.float()
    g = x.view(x.shape[0], -1, 128)
    amax = g.abs().amax(-1)
    if divide:
        # by a tensor: a division by a number multiplies by its reciprocal, which moves exact ties
        scale = (amax / torch.full_like(amax, 448.0)).clamp_min(torch.finfo(torch.float32).tiny)
        v = g / scale[..., None]
    else:
        scale = amax.clamp_min(1e-10) * torch.tensor(1.0 / 448.0, device=x.device)
        v = g * (1.0 / scale)[..., None]
    return v.clamp(-448.0, 448.0).to(torch.float8_e4m3fn).float(), scale


def _dequantized_rows(x, divide=False):
    v, scale = _groups_fp8(x, divide)
    return (v.to(F64) * scale.to(F64)[..., None]).view(x.shape)


def _dequantized_weight(codes, scales):
    n, k = codes.shape
    return codes.float().to(F64) * scales.to(F64).repeat_interleave(128, 0)[:n].repeat_interleave(128, 1)


def _by_columns(rows, n, weight_rows):
    """rows @ weight^T, the weight decoded 8192 rows at a time."""
    return torch.cat([rows @ weight_rows(r, min(n, r + 8192)).t() for r in range(0, n, 8192)], 1)


_E2M1 = (0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0)


def _dequantized_mxfp4(codes, scales):
    lut = torch.tensor(_E2M1 + tuple(-v for v in _E2M1), dtype=F64, device=codes.device)
    values = torch.stack((lut[(codes & 15).long()], lut[(codes >> 4).long()]), -1).view(codes.shape[0], -1)
    return values * torch.exp2(scales.to(F64) - 127).repeat_interleave(32, 1)


def _mxfp4_rows(x):
    """MXFP4 activations decoded: the exponent that brings a block's largest value to at most 6, then the
    nearest of the e2m1 values, ties to the even code."""
    g = x.to(F64).view(x.shape[0], -1, 32)
    mant, expo = torch.frexp(g.abs().amax(-1).clamp_min(1e-10))
    scale = torch.exp2((expo - 3 + (mant > 0.75).int()).clamp(-127, 127).to(F64))[..., None]
    v = (g / scale).abs()
    step = torch.where(v < 2, 0.5, torch.where(v < 4, 1.0, 2.0))
    return (torch.round(v / step) * step * torch.sign(g) * scale).view(x.shape)


def _first_largest(values, k):
    return torch.sort(values, dim=-1, descending=True, stable=True).indices[:, :k]


def _route(logits, bias, groups, kept):
    scores = torch.sigmoid(logits.to(F64))
    biased = scores + bias.to(F64)
    t, e = biased.shape
    best = torch.topk(biased.view(t, groups, -1), 2).values.sum(-1)
    allowed = torch.zeros_like(best, dtype=torch.bool).scatter_(1, _first_largest(best, kept), True)
    masked = torch.where(allowed.repeat_interleave(e // groups, 1), biased, float("-inf"))
    ids = _first_largest(masked, TOPK)
    weights = scores.gather(1, ids)
    weights = 2.5 * weights / weights.sum(1, keepdim=True)
    shared = torch.ones((t, 1), dtype=F64, device=ids.device)
    return torch.cat((ids, e * shared.long()), 1), torch.cat((weights, shared), 1)


def _mlp(x, w1, s1, w2, s2):
    gate, up = (_dequantized_rows(x, True) @ _dequantized_weight(w1, s1).t()).chunk(2, 1)
    h = (gate * torch.sigmoid(gate) * up).to(torch.bfloat16)
    return _dequantized_rows(h, True) @ _dequantized_weight(w2, s2).t()


def _exact_experts(x, ids, weights, w1, s1, w2, s2):
    out = torch.zeros(x.shape, dtype=F64, device=x.device)
    for e in range(w1.shape[0]):
        tokens, slots = torch.nonzero(ids == e, as_tuple=True)
        if tokens.numel():
            y = _mlp(x[tokens], w1[e], s1[e], w2[e], s2[e])
            out.index_add_(0, tokens, y * weights[tokens, slots][:, None])
    return out


def exact(case, seed):
    op = case["op"]
    if op == "quant_fp8":
        v, scale = _groups_fp8(_activations(case, seed), False)
        return v.reshape(case["m"], case["k"]).to(F64), scale.t().contiguous().to(F64)
    if op == "quant_mxfp8":
        g = _activations(case, seed).float().view(case["m"], -1, 32)
        raw = (g.abs().amax(-1).clamp_min(1e-10) * torch.tensor(1.0 / 448.0, device=DEV)).view(torch.int32)
        expo = (raw >> 23) + ((raw & 0x7FFFFF) != 0).int()
        v = (g / torch.exp2(expo.float() - 127)[..., None]).clamp(-448.0, 448.0).to(torch.float8_e4m3fn)
        return v.float().reshape(case["m"], case["k"]).to(F64), expo.to(torch.uint8)
    if op in ("linear_fp8", "fused_fp8", "gemm_fp8"):
        b, bs = _fp8_weight(case, seed)
        rows = _dequantized_rows(_activations(case, seed))
        out = _by_columns(rows, case["n"], lambda r, e: _dequantized_weight(b[r:e], bs[r // 128:-(-e // 128)]))
        bias = _bias(case, seed)
        return out if bias is None else out + bias.to(F64)
    if op == "linear_mxfp4":
        b, bs = _mxfp4_weight(case, seed)
        return _by_columns(_mxfp4_rows(_activations(case, seed)), case["n"],
                           lambda r, e: _dequantized_mxfp4(b[r:e], bs[r:e]))
    w1, s1, w2, s2 = _experts(case, seed)
    if op == "moe_layer":
        x, router, correction = _router(case, seed)
        logits = (x.to(F64) @ router.to(F64).t()).to(torch.bfloat16)
        ids, weights = _route(logits, correction, 8, 4)
        return _exact_experts(x, ids, weights, w1, s1, w2, s2)
    ids, weights = _route(*_logits(case, seed), 1, 1)
    return {"ids": None, "weights": weights,
            "out": _exact_experts(_activations(case, seed), ids, weights, w1, s1, w2, s2)}
