"""The work this framework is measured on: whole passes through its public operators, at the sizes it is used at.

A case is one of three kinds.

  layer       one MoE layer on one GPU: calc_scatter_index -> GemmGroupedV3AGScatter.forward (or
              forward_multiple_weights and a SiLU gate) -> [fp8: Quantization.quantize_rowwise] ->
              GemmGroupedV3GatherRS.forward_gather_rs, in bf16, fp16 or fp8
  blockscale  one GPU's experts with block-scaled fp8 on rows that are already grouped by expert:
              quantize_vector_blockwise -> BlockScaleGemm.forward_grouped, twice, then topk_weighted_gather_reduce
  quant       one tensor quantised to e4m3, with or without the transposed copy that a backward pass reads

Activations are N(0, 1), weights N(0, 0.02), routing either the top-k of N(0, 1) logits, uniform, or Zipf with exponent
1.2.  Token counts run from one token being decoded to a whole prefill batch; the operators are built once, as a
program keeps them.
"""
import math

import torch

import flux_amd

E4M3_MAX = 448.0
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "fp8": torch.float8_e4m3fn}


def _layer(name, dtype, tokens, topk, experts, hidden, ffn, routing="softmax", gated=False):
    return {"name": name, "kind": "layer", "dtype": dtype, "tokens": tokens, "topk": topk, "experts": experts,
            "hidden": hidden, "ffn": ffn, "routing": routing, "gated": gated}


def listed():
    return [
        # A small layer: 256 tokens, 8 experts.  Launches and host time are most of it.
        _layer("small_bf16", "bf16", 256, 2, 8, 1024, 2048),
        # One user decoding one token with eight large experts: two experts' weights are read for one row each.
        _layer("decode_one_bf16", "bf16", 1, 2, 8, 4096, 14336),
        # A small decode batch on the same layer: every expert is hit by a handful of rows.
        _layer("decode_batch_bf16", "bf16", 37, 2, 8, 4096, 14336),
        # Decoding with many small experts and a gated activation (gate and up projections in one call).
        _layer("decode_fine_bf16", "bf16", 96, 6, 64, 2048, 1408, gated=True),
        # Decoding with fp8 weights, one GPU's share of a wide layer.
        _layer("decode_fp8", "fp8", 128, 8, 32, 7168, 2048, routing="uniform"),
        # A chunk of a prefill between the two regimes, in fp16, at a token count no tile divides.
        _layer("chunk_f16", "f16", 777, 2, 8, 4096, 14336),
        # A whole prefill batch over eight large experts.
        _layer("prefill_bf16", "bf16", 8192, 2, 8, 4096, 14336),
        # Prefill over many small experts with a skewed load: some experts get thousands of rows, some a few.
        _layer("prefill_zipf_bf16", "bf16", 16384, 6, 64, 2048, 1408, routing="zipf"),
        # Prefill with fp8 weights and activations.
        _layer("prefill_fp8", "fp8", 4096, 8, 32, 7168, 2048, routing="uniform"),
        # Block-scaled fp8 experts, a decode batch and a prefill batch.
        {"name": "decode_blockscale", "kind": "blockscale", "tokens": 50, "topk": 8, "experts": 32, "hidden": 7168,
         "ffn": 2048, "routing": "uniform"},
        {"name": "prefill_blockscale", "kind": "blockscale", "tokens": 2048, "topk": 8, "experts": 32, "hidden": 7168,
         "ffn": 2048, "routing": "uniform"},
        # Activations of a training step quantised for forward and backward (both directions from one tensor).
        {"name": "quant_train", "kind": "quant", "method": "vector_t", "rows": 11000, "cols": 7168},
    ]


# ---- inputs ---------------------------------------------------------------------------------------------------


def _choose_experts(routing, tokens, topk, experts, gen):
    """[tokens, topk] int32 expert ids and fp32 weights that sum to one."""
    logits = torch.randn(tokens, experts, generator=gen, device="cuda")
    if routing == "softmax":
        weight, idx = torch.topk(torch.softmax(logits, dim=-1), topk, dim=-1)
    else:  # without replacement from a fixed distribution: the top-k of log p + Gumbel noise
        logp = torch.zeros(experts, device="cuda")
        if routing == "zipf":
            logp = -1.2 * torch.log(torch.arange(1, experts + 1, device="cuda", dtype=torch.float32))
        u = torch.rand(tokens, experts, generator=gen, device="cuda").clamp_(1e-9, 1 - 1e-7)
        idx = torch.topk(logp - torch.log(-torch.log(u)), topk, dim=-1).indices
        weight = torch.softmax(torch.gather(logits, 1, idx), dim=-1)
    weight = weight / weight.sum(dim=-1, keepdim=True)
    return idx.to(torch.int32).contiguous(), weight


def _route(case, gen):
    tokens, topk, experts = case["tokens"], case["topk"], case["experts"]
    choosed, weight = _choose_experts(case["routing"], tokens, topk, experts, gen)
    flat = choosed.flatten().long()
    order = torch.argsort(flat, stable=True)
    scatter = torch.empty_like(order)
    scatter[order] = torch.arange(order.numel(), device="cuda")
    splits = torch.bincount(flat, minlength=experts).to(torch.int32)
    return {"choosed": choosed, "splits": splits, "splits_cpu": splits.cpu(),
            "routing_idx": scatter.to(torch.int32), "row_weight": weight.flatten()[order].contiguous()}


def _weights(experts, n, k, dtype, gen):
    """[E, N, K] N(0, 0.02)."""
    w = torch.empty(experts, n, k, device="cuda", dtype=dtype)
    for e in range(experts):
        w[e] = torch.randn(n, k, generator=gen, device="cuda") * 0.02
    return w


def _fp8_weights(experts, n, k, scales, gen):
    """[E, N, K] e4m3 and fp32 scales: one per expert, per output channel, or per 128 x 128 block."""
    q = torch.empty(experts, n, k, device="cuda", dtype=torch.float8_e4m3fn)
    out = []
    for e in range(experts):
        w = torch.randn(n, k, generator=gen, device="cuda") * 0.02
        if scales == "expert":
            s = w.abs().amax() / E4M3_MAX
            q[e] = (w / s).to(torch.float8_e4m3fn)
        elif scales == "channel":
            s = w.abs().amax(dim=1) / E4M3_MAX
            q[e] = (w / s[:, None]).to(torch.float8_e4m3fn)
        else:
            b = w.view(n // 128, 128, k // 128, 128)
            s = b.abs().amax(dim=(1, 3)) / E4M3_MAX
            q[e] = (b / s[:, None, :, None]).view(n, k).to(torch.float8_e4m3fn)
        out.append(s)
    return q, torch.stack(out).contiguous()


def _prepare_layer(case, gen):
    t, k, e, h, f = (case[n] for n in ("tokens", "topk", "experts", "hidden", "ffn"))
    dtype = DTYPES[case["dtype"]]
    s = _route(case, gen)
    x = torch.randn(t, h, generator=gen, device="cuda")
    s["gated"], s["output_scale"], s["weight_scale"], s["quant"] = case["gated"], None, None, None
    groups = 2 if case["gated"] else 1
    if case["dtype"] == "fp8":
        # layer0: one scale for the activations, one per expert for the weights; layer1: per row and per output channel
        sx = x.abs().amax() / E4M3_MAX
        s["x"] = (x / sx).to(dtype)
        pairs = [_fp8_weights(e, f, h, "expert", gen) for _ in range(groups)]
        s["w1"] = [q for q, _ in pairs]
        s["output_scale"] = [(sw * sx).contiguous() for _, sw in pairs]
        s["w2"], s["weight_scale"] = _fp8_weights(e, h, f, "channel", gen)
        s["quant"] = flux_amd.Quantization(torch.bfloat16, torch.float8_e4m3fn)
    else:
        s["x"] = x.to(dtype)
        s["w1"] = [_weights(e, f, h, dtype, gen) for _ in range(groups)]
        s["w2"] = _weights(e, h, f, dtype, gen)
    s["op0"] = flux_amd.GemmGroupedV3AGScatter(flux_amd.DistEnvTPWithEP(None, 1, None),
                                               flux_amd.MoeArguments(t, h, f, e, k, dtype))
    s["op1"] = flux_amd.GemmGroupedV3GatherRS(e, t * k, h, k, 0, 1, 1, 1)
    return s


def _run_layer(s):
    scatter = flux_amd.calc_scatter_index(s["choosed"], s["splits"])
    if s["gated"]:
        gate, up = s["op0"].forward_multiple_weights(s["x"], s["w1"], s["splits"], scatter, output_scale=s["output_scale"])
        y = torch.nn.functional.silu(gate) * up
    else:
        y = s["op0"].forward(s["x"], s["w1"][0], s["splits"], scatter,
                             output_scale=s["output_scale"][0] if s["output_scale"] else None)
    act, row_scale = (y, None) if s["quant"] is None else s["quant"].quantize_rowwise(y)
    out = s["op1"].forward_gather_rs(act, s["w2"], s["splits_cpu"], scatter.view(-1), input_scale=row_scale,
                                     weight_scale=s["weight_scale"], output_vec_scale=s["row_weight"])
    return {"scatter": scatter, "y": y, "out": out}


def _prepare_blockscale(case, gen):
    t, k, e, h, f = (case[n] for n in ("tokens", "topk", "experts", "hidden", "ffn"))
    s = _route(case, gen)
    s["topk"] = k
    s["rows"] = torch.randn(t * k, h, generator=gen, device="cuda").to(torch.bfloat16)  # grouped by expert
    s["w1"], s["w1_scale"] = _fp8_weights(e, f, h, "block", gen)
    s["w2"], s["w2_scale"] = _fp8_weights(e, h, f, "block", gen)
    s["quant"] = flux_amd.Quantization(torch.bfloat16, torch.float8_e4m3fn)
    s["gemm"] = flux_amd.BlockScaleGemm(torch.float8_e4m3fn, torch.float8_e4m3fn, torch.bfloat16)
    return s


def _run_blockscale(s):
    qx, sx, _, _ = s["quant"].quantize_vector_blockwise(s["rows"], return_tranpose=False)
    y = s["gemm"].forward_grouped(qx, s["splits_cpu"], s["w1"], input_scale=sx, weight_scale=s["w1_scale"])
    qy, sy, _, _ = s["quant"].quantize_vector_blockwise(y, return_tranpose=False)
    z = s["gemm"].forward_grouped(qy, s["splits_cpu"], s["w2"], input_scale=sy, weight_scale=s["w2_scale"])
    out = flux_amd.topk_weighted_gather_reduce([z], s["routing_idx"], s["topk"], s["row_weight"])
    return {"y": y, "z": z, "out": out}


def _prepare_quant(case, gen):
    x = torch.randn(case["rows"], case["cols"], generator=gen, device="cuda")
    # a few outlier channels, as activations have them
    x[:, :: 97] *= 8.0
    return {"x": x.to(torch.bfloat16), "method": case["method"],
            "quant": flux_amd.Quantization(torch.bfloat16, torch.float8_e4m3fn)}


def _run_quant(s):
    x, q = s["x"], s["quant"]
    if s["method"] == "rowwise":
        codes, scale = q.quantize_rowwise(x)
        return {"q": codes.view(torch.uint8), "scale": scale}
    transpose = s["method"].endswith("_t")
    call = q.quantize_vector_blockwise if s["method"].startswith("vector") else q.quantize_square_blockwise
    codes, scale, codes_t, scale_t = call(x, return_tranpose=transpose)
    out = {"q": codes.view(torch.uint8), "scale": scale}
    if transpose:
        out.update(q_t=codes_t.view(torch.uint8), scale_t=scale_t)
    return out


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    make = {"layer": _prepare_layer, "blockscale": _prepare_blockscale, "quant": _prepare_quant}[case["kind"]]
    state = make(case, gen)
    state["kind"] = case["kind"]
    return state


def run(state):
    return {"layer": _run_layer, "blockscale": _run_blockscale, "quant": _run_quant}[state["kind"]](state)


# ---- what a pass cannot do without ------------------------------------------------------------------------------


def _experts_hit(case):
    """Expected number of experts with at least one row."""
    t, k, e = case["tokens"], case["topk"], case["experts"]
    if case["routing"] == "zipf":
        p = [(i + 1) ** -1.2 for i in range(e)]
        share = [min(1.0, k * v / sum(p)) for v in p]
    else:
        share = [k / e] * e
    return sum(1.0 - (1.0 - s) ** t for s in share)


def work(case):
    """Inputs of every call read once, its results written once, the weights of the experts that are hit read once."""
    if case["kind"] == "quant":
        r, c = case["rows"], case["cols"]
        copies = 2 if case["method"].endswith("_t") else 1
        scales = {"rowwise": r, "vector": r * (c // 128), "square": r * c // 16384}[case["method"].split("_")[0]]
        return {"bytes": r * c * (2 + copies) + scales * copies * 4, "flops": 0}
    t, k, h, f = (case[n] for n in ("tokens", "topk", "hidden", "ffn"))
    m, hit = t * k, _experts_hit(case)
    if case["kind"] == "blockscale":
        weights = 2 * hit * h * f
        rows = m * h * (2 + 1 + 1) + m * f * (2 + 2 + 1 + 1) + m * h * (2 + 2) + m * (h + f) // 128 * 8
        return {"bytes": weights + rows + t * h * 2 + m * 8, "flops": 4 * m * h * f}
    groups = 2 if case["gated"] else 1
    elt = 1 if case["dtype"] == "fp8" else 2
    weights = (groups + 1) * hit * h * f * elt
    rows = t * h * elt + groups * m * f * 2 + m * f * elt + t * h * 2
    if case["gated"]:
        rows += (groups + 1) * m * f * 2
    if case["dtype"] == "fp8":
        rows += m * f * (2 + 1)
    return {"bytes": weights + rows + m * 16, "flops": 2 * (groups + 1) * m * h * f}


def tolerance(case):
    """About four times what summing K in another order changes: 3.6e-4 in bf16, 9e-5 in fp16, 1.6e-3 in fp8 and 1.4e-3
    block-scaled, where a rounding of the first product that falls the other way moves an e4m3 code of the second's input."""
    if case["kind"] == "quant":
        return "exact"
    if case["kind"] == "blockscale":
        return {"rel": 6e-3}
    return {"rel": {"bf16": 1.5e-3, "f16": 4e-4, "fp8": 6e-3}[case["dtype"]]}


# ---- drawn cases ------------------------------------------------------------------------------------------------


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_once(rng):
    kind = rng.choices(["layer", "blockscale", "quant"], [6, 2, 2])[0]
    if kind == "quant":
        return {"kind": kind, "method": rng.choice(["rowwise", "vector", "vector_t", "square_t"]),
                "rows": _log_int(rng, 16, 32768), "cols": 16 * rng.randint(64, 512)}
    topk = rng.choice([1, 2, 2, 3, 4, 6, 8])
    case = {"kind": kind, "tokens": _log_int(rng, 1, 16384), "topk": topk, "experts": _log_int(rng, max(4, topk), 96),
            "hidden": 128 * rng.randint(8, 56), "ffn": 128 * _log_int(rng, 6, 112),
            "routing": rng.choice(["softmax", "uniform", "zipf"])}
    if kind == "layer":
        case["dtype"] = rng.choices(["bf16", "f16", "fp8"], [5, 2, 3])[0]
        case["gated"] = rng.random() < 0.3
        if rng.random() < 0.3:  # widths that are not whole tiles
            case["hidden"] -= 16 * rng.randint(1, 7)
            case["ffn"] -= 16 * rng.randint(1, 7)
    return case


def draw(rng):
    """One more case of the same ranges, at most half the arithmetic and no more bytes than the largest listed case."""
    largest = [work(c) for c in listed()]
    bytes_, flops = max(w["bytes"] for w in largest), max(w["flops"] for w in largest) / 2
    while True:
        case = _draw_once(rng)
        w = work(case)
        store = 0 if case["kind"] == "quant" else 3 * case["experts"] * case["hidden"] * case["ffn"] * (
            1 if case["kind"] == "blockscale" or case["dtype"] == "fp8" else 2)
        if w["bytes"] <= bytes_ and w["flops"] <= flops and store <= 6e9:
            return case
