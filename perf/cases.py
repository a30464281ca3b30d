"""Performance cases of the library: what a serving program has it do, through the public entry points.

Four families, each over its whole range of sizes:

  gemm     one linear layer through ``compile_preshuffle_gemm`` (fp8 / int8 with per-token and per-channel scales, bf16 / fp16
           without), with or without the activation quantiser in front, with every fused epilogue;
  mx       one linear layer through the MX ``launch_gemm`` (fp4 / fp6 / fp8 activations, fp4 / fp8 weights), fp4
           activations with or without the quantiser in front;
  moe      one MoE layer of the 2-stage pair (fp8, int8 or int8 activations with int4 weights): quantise, gate and sort,
           gate-up stage, quantise, down stage (accumulating, or one row per slot and a reduction);
  moe_mx   one MoE layer of the fused MX-FP4 pair: quantise (or let stage 1 do it), gate and sort, both stages.

The listed cases are the shapes this repository's benchmark and tests are about; ``draw`` gives others of the same ranges.
"""

from __future__ import annotations

import math

import torch

from flydsl_amd import layout, quant, quant_device
from flydsl_amd.kernels.gemm.mxfp4_preshuffle import launch_gemm
from flydsl_amd.kernels.gemm.preshuffle_gemm import compile_preshuffle_gemm
from flydsl_amd.kernels.moe.moe_gemm_2stage import compile_moe_gemm1, compile_moe_gemm2, compile_moe_reduction
from flydsl_amd.kernels.moe.moe_sorting import moe_softmax_sort_flydsl, moe_sorting_get_workspace_size, sorted_sizes
from flydsl_amd.kernels.moe.mxfp_moe import flydsl_mxfp4_gemm1, flydsl_mxfp4_gemm2, moe_mxfp4_sort

TORCH_OUT = {"bf16": torch.bfloat16, "fp16": torch.float16, "f16": torch.float16}
QUANT = {"fp8": torch.float8_e4m3fn, "int8": torch.int8, "int4": torch.int8}


def listed():
    return [
        # single-stream decode of one projection, activations already quantised by the layer before: the smallest call, where
        # launching and one pass over the weight are everything
        dict(name="fp8_decode_m16", kind="gemm", dtype="fp8", out="bf16", M=16, N=6144, K=4096, epilogue="none", quantize=False),
        # continuous batching: a couple of hundred rows, not a multiple of anything, against a large weight
        dict(name="fp8_batch_m200", kind="gemm", dtype="fp8", out="bf16", M=200, N=8192, K=8192, epilogue="bias_silu", quantize=True),
        # prefill of a whole prompt with the quantiser in front
        dict(name="fp8_prefill_m8192", kind="gemm", dtype="fp8", out="bf16", M=8192, N=4096, K=4096, epilogue="none", quantize=True),
        # the widest feed-forward layer, int8
        dict(name="int8_ffn_m4096", kind="gemm", dtype="int8", out="bf16", M=4096, N=28672, K=8192, epilogue="none", quantize=False),
        # an unquantised layer on a ragged number of rows with a fused activation
        dict(name="bf16_m5133_gelu", kind="gemm", dtype="bf16", out="bf16", M=5133, N=5120, K=8320, epilogue="bias_gelu", quantize=False),
        # MXFP4 decode and prefill of one projection, quantiser in front
        dict(name="mxfp4_decode_m32", kind="mx", a="fp4", b="fp4", out="bf16", M=32, N=7168, K=2048, batch=1, quantize=True),
        dict(name="mxfp4_prefill_m4096", kind="mx", a="fp4", b="fp4", out="bf16", M=4096, N=7168, K=2048, batch=1, quantize=True),
        # mixed MX formats (fp8 activations for accuracy, fp4 weights) on a decode batch
        dict(name="mx_a8w4_m64", kind="mx", a="fp8", b="fp4", out="bf16", M=64, N=8192, K=8192, batch=1, quantize=False),
        # one MoE layer: a decode batch, bound by the experts' weights, and a prefill batch, bound by the matrix cores
        dict(name="moe_fp8_decode_t64", kind="moe", dtype="fp8", out="bf16", tokens=64, model=4096, inter=1536, experts=32, topk=8, block=16, accumulate=True),
        dict(name="moe_fp8_prefill_t4096", kind="moe", dtype="fp8", out="bf16", tokens=4096, model=4096, inter=1536, experts=32, topk=8, block=128, accumulate=True),
        # the same two in MX-FP4
        dict(name="moe_mxfp4_decode_t64", kind="moe_mx", out="bf16", tokens=64, model=4096, inter=1536, experts=32, topk=8, block=32, inline=False),
        dict(name="moe_mxfp4_prefill_t4096", kind="moe_mx", out="bf16", tokens=4096, model=4096, inter=1536, experts=32, topk=8, block=128, inline=False),
    ]


def _log(rng, lo, hi, step=1):
    """A multiple of `step` between lo and hi, spread over the logarithm."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(step, int(round(v / step)) * step)


def _draw_gemm(rng):
    dtype = rng.choice(["fp8", "fp8", "fp8", "int8", "int8", "bf16", "fp16"])
    wide = dtype in ("bf16", "fp16")
    n, k = _log(rng, 1024, 28672, 16), _log(rng, 1024, 8320 if wide else 14336, 64)
    # at most the work of the largest listed layers (1.9e12 operations in 8 bits, 0.44e12 in 16)
    m = min(_log(rng, 1, 8192), max(1, int((0.44e12 if wide else 1.9e12) / (2.0 * n * k))))
    return dict(kind="gemm", dtype=dtype, out=rng.choice(["bf16", "bf16", "fp16"]), M=m, N=n, K=k,
                epilogue=rng.choice(["none", "none", "none", "bias", "bias_relu", "bias_silu", "bias_gelu"]),
                quantize=not wide and rng.random() < 0.5)


def _draw_mx(rng):
    a, b = rng.choice([("fp4", "fp4"), ("fp4", "fp4"), ("fp4", "fp4"), ("fp8", "fp8"), ("fp8", "fp4"), ("fp6", "fp4")])
    batch = 1 if rng.random() < 0.85 else rng.randint(2, 4)
    n, k = _log(rng, 1024, 16384, 32), _log(rng, 1024, 14336, 256)
    general = batch > 1 or (a, b) != ("fp4", "fp4")
    m = min(_log(rng, 1, 8192), max(1, int((0.4e12 if general else 0.8e12) / (2.0 * n * k * batch))))
    return dict(kind="mx", a=a, b=b, out=rng.choice(["bf16", "bf16", "fp16"]), M=m, N=n, K=k, batch=batch,
                quantize=(a, b, batch) == ("fp4", "fp4", 1) and rng.random() < 0.5)


def _draw_moe(rng, mx):
    experts = rng.choice([8, 16, 17, 32, 64, 128])
    topk = rng.choice([1, 2, 4, 6, 8])
    model, inter = 256 * rng.randint(4, 16), 256 * rng.randint(1, 8)
    while experts * model * inter > 32 * 4096 * 1536:  # the experts' weights of the listed layers are the most
        experts //= 2
    tokens = min(_log(rng, 1, 4096), max(1, int(4096 * 8 * 4096 * 1536 / (topk * model * inter))))
    rows = tokens * topk / experts  # routed rows per expert decide the block of the sorted list, as in the tests
    block = 16 if rows <= 24 else 32 if rows <= 48 else 64 if rows <= 96 else 128
    if not mx:
        return dict(kind="moe", dtype=rng.choice(["fp8", "fp8", "int8", "int4"]), out=rng.choice(["bf16", "f16"]), tokens=tokens, model=model,
                    inter=inter, experts=experts, topk=topk, block=block, accumulate=rng.random() < 0.7)
    inline = block == 16 and rng.random() < 0.5
    return dict(kind="moe_mx", out=rng.choice(["bf16", "f16"]), tokens=tokens, model=model, inter=inter, experts=experts, topk=topk,
                block=16 if inline else max(32, block), inline=inline)


def draw(rng):
    family = rng.choice(["gemm"] * 5 + ["mx"] * 3 + ["moe"] * 3 + ["moe_mx"])
    if family == "gemm":
        return _draw_gemm(rng)
    if family == "mx":
        return _draw_mx(rng)
    return _draw_moe(rng, family == "moe_mx")


# ---- inputs: activations N(0, 1), weights N(0, 0.02), router logits N(0, 1), all made on the GPU from the seed ----


def _randn(g, *shape, std=1.0, dtype=torch.bfloat16):
    return torch.randn(*shape, generator=g, device="cuda", dtype=dtype).mul_(std)


def _quant_weight(g, rows, k, dtype):
    """Quantised, preshuffled weight of `rows` x k (flat bytes) and its scale per row."""
    w = _randn(g, rows, k, std=0.02)
    q, s = quant_device.pertoken_quant(w, quant_dtype=QUANT[dtype])
    return layout.shuffle_weight(q.view(torch.int8)).view(QUANT[dtype]).contiguous(), s.view(-1).contiguous()


def _quant_mx_weight(g, rows, k, fmt):
    """MX-quantised, preshuffled weight of `rows` x k and its shuffled scales."""
    w = _randn(g, rows, k, std=0.02)
    if fmt == "fp4":
        codes, scales = quant_device.per_1x32_f4_quant(w, shuffle=True)
        scales = scales.view(torch.uint8)
    else:
        codes, scales = quant.per_1x32_f8_quant(w)
        scales = layout.shuffle_scale_w4(scales.view(torch.uint8))
    return layout.shuffle_weight_w4(codes.view(torch.uint8)).contiguous(), scales.contiguous()


def _prepare_gemm(c, g):
    m, n, k, dtype = c["M"], c["N"], c["K"], c["dtype"]
    s = {"case": c, "M": m, "N": n, "stream": torch.cuda.current_stream()}
    out = TORCH_OUT[c["out"]]
    if dtype in ("bf16", "fp16"):
        td = TORCH_OUT[dtype]
        s["a"] = _randn(g, m, k).to(td)
        s["b"] = layout.shuffle_weight(_randn(g, n, k, std=0.02).to(td)).contiguous()
        s["sa"] = s["sb"] = None
    else:
        s["b"], s["sb"] = _quant_weight(g, n, k, dtype)
        x = _randn(g, m, k)
        s["x"] = x if c["quantize"] else None
        s["a"], s["sa"] = quant_device.pertoken_quant(x, quant_dtype=QUANT[dtype])
    s["bias"] = _randn(g, n, std=0.1).to(out) if c["epilogue"] != "none" else torch.empty(0, dtype=out, device="cuda")
    s["c"] = torch.empty(m, n, dtype=out, device="cuda")
    s["fn"] = compile_preshuffle_gemm(N=n, K=k, tile_m=128, tile_n=256, tile_k=64, in_dtype=dtype, out_dtype=c["out"], epilogue=c["epilogue"])
    return s


def _run_gemm(s):
    if s.get("x") is not None:
        quant_device.pertoken_quant(s["x"], quant_dtype=QUANT[s["case"]["dtype"]], stream=s["stream"], out=(s["a"], s["sa"]))
    s["fn"](s["c"], s["a"], s["b"], s["sa"], s["sb"], s["bias"], s["M"], s["N"], s["stream"])
    return s["c"]


def _prepare_mx(c, g):
    m, n, k, batch = c["M"], c["N"], c["K"], c["batch"]
    s = {"case": c, "stream": torch.cuda.current_stream()}
    s["b"], s["sb"] = _quant_mx_weight(g, batch * n, k, c["b"])
    x = _randn(g, batch, m, k)
    if batch == 1 and c["a"] == "fp4":
        s["x"] = x[0] if c["quantize"] else None
        s["a"], s["sa"] = quant_device.per_1x32_f4_quant(x[0], shuffle=True)
    else:
        m32 = (m + 31) // 32 * 32  # the scales of every batch cover whole 32-row chunks
        xp = torch.zeros(batch * m32, k, device="cuda")
        xp.view(batch, m32, k)[:, :m] = x
        q = {"fp4": quant.per_1x32_f4_quant, "fp6": quant.per_1x32_f6_quant, "fp8": quant.per_1x32_f8_quant}[c["a"]](xp)
        codes = q[0].view(torch.uint8)
        s["a"] = codes.view(batch, m32, -1)[:, :m].contiguous()
        s["sa"] = layout.shuffle_scale_w4(q[1].view(torch.uint8)).contiguous()
    s["c"] = torch.empty(batch, m, n, dtype=TORCH_OUT[c["out"]], device="cuda")
    return s


def _run_mx(s):
    c = s["case"]
    if s.get("x") is not None:
        quant_device.per_1x32_f4_quant(s["x"], shuffle=True, stream=s["stream"], out=(s["a"], s["sa"]))
    launch_gemm(s["c"], s["a"], s["b"], s["sa"], s["sb"], c["M"], c["N"], s["stream"], c["N"], c["K"], 64, 256, 256, c["a"], c["out"], c["b"],
                c["batch"], -1, -1, -1, -1, -1, -1, 0, 0)
    return s["c"]


def _prepare_routing(c, g):
    tokens, experts, topk = c["tokens"], c["experts"], c["topk"]
    s = {"case": c, "stream": torch.cuda.current_stream()}
    s["x"] = _randn(g, tokens, c["model"])
    s["logits"] = _randn(g, tokens, experts)
    rows, blocks = sorted_sizes(tokens, topk, experts, c["block"])
    s["sid"] = torch.empty(rows, dtype=torch.int32, device="cuda")
    s["swt"] = torch.empty(rows, dtype=torch.float32, device="cuda")
    s["se"] = torch.empty(blocks, dtype=torch.int32, device="cuda")
    s["nv"] = torch.empty(2, dtype=torch.int32, device="cuda")
    s["ids"] = torch.empty(tokens, topk, dtype=torch.int32, device="cuda")
    s["wts"] = torch.empty(tokens, topk, dtype=torch.float32, device="cuda")
    size = moe_sorting_get_workspace_size(tokens, experts, topk)
    s["ws"] = torch.empty(size, dtype=torch.uint8, device="cuda") if size else None
    s["rows"], s["blocks"] = rows, blocks
    s["out"] = torch.empty(tokens, c["model"], dtype=TORCH_OUT[c["out"]], device="cuda")
    return s


def _route(s, clear):
    c = s["case"]
    moe_softmax_sort_flydsl(s["logits"], s["sid"], s["swt"], s["se"], s["nv"], clear, c["experts"], c["topk"], "bf16", c["block"], None, True, None,
                            topk_ids=s["ids"], topk_weights=s["wts"], workspace=s["ws"], stream=s["stream"])


def _prepare_moe(c, g):
    s = _prepare_routing(c, g)
    tokens, model, inter, experts, topk, dtype = c["tokens"], c["model"], c["inter"], c["experts"], c["topk"], c["dtype"]
    if dtype == "int4":
        w = torch.randint(-8, 8, (experts * 2 * inter, model), generator=g, device="cuda", dtype=torch.int8)
        s["w1"] = layout.pack_shuffled_int8_to_int4(layout.shuffle_weight(w))
        w = torch.randint(-8, 8, (experts * model, inter), generator=g, device="cuda", dtype=torch.int8)
        s["w2"] = layout.pack_shuffled_int8_to_int4(layout.shuffle_weight(w))
        s["sw1"] = torch.rand(experts * 2 * inter, generator=g, device="cuda").mul_(0.004).add_(0.002)
        s["sw2"] = torch.rand(experts * model, generator=g, device="cuda").mul_(0.004).add_(0.002)
    else:
        s["w1"], s["sw1"] = _quant_weight(g, experts * 2 * inter, model, dtype)
        s["w2"], s["sw2"] = _quant_weight(g, experts * model, inter, dtype)
    td, qd = TORCH_OUT[c["out"]], QUANT[dtype]
    s["xq"] = torch.empty(tokens, model, dtype=qd, device="cuda")
    s["sx"] = torch.empty(tokens, 1, dtype=torch.float32, device="cuda")
    s["h"] = torch.empty(tokens * topk, inter, dtype=td, device="cuda")
    s["hq"] = torch.empty(tokens * topk, inter, dtype=qd, device="cuda")
    s["sh"] = torch.empty(tokens * topk, 1, dtype=torch.float32, device="cuda")
    kw = dict(model_dim=model, inter_dim=inter, experts=experts, topk=topk, tile_m=c["block"], tile_n=128, tile_k=128, out_dtype=c["out"], in_dtype=dtype)
    s["stage1"] = compile_moe_gemm1(doweight_stage1=False, **kw)
    s["stage2"] = compile_moe_gemm2(doweight_stage2=True, accumulate=c["accumulate"], **kw)
    if not c["accumulate"]:
        s["slots"] = torch.empty(tokens, topk, model, dtype=td, device="cuda")
        s["reduce"] = compile_moe_reduction(topk=topk, model_dim=model, dtype_str=c["out"])
    return s


def _run_moe(s):
    c, st = s["case"], s["stream"]
    tokens, model, inter, qd = c["tokens"], c["model"], c["inter"], QUANT[c["dtype"]]
    quant_device.pertoken_quant(s["x"], quant_dtype=qd, stream=st, out=(s["xq"], s["sx"]))
    _route(s, s["out"] if c["accumulate"] else None)
    s["stage1"](s["h"], s["xq"], s["w1"], s["sx"], s["sw1"], s["sid"], s["se"], s["swt"], s["nv"], tokens, inter, model, s["blocks"], st)
    quant_device.pertoken_quant(s["h"], quant_dtype=qd, stream=st, out=(s["hq"], s["sh"]))
    if c["accumulate"]:
        s["stage2"](s["out"], s["hq"], s["w2"], s["sh"], s["sw2"], s["sid"], s["se"], s["swt"], s["nv"], tokens, model, inter, s["blocks"], st)
    else:
        s["stage2"](s["slots"], s["hq"], s["w2"], s["sh"], s["sw2"], s["sid"], s["se"], s["swt"], s["nv"], tokens, model, inter, s["blocks"], st)
        s["reduce"](s["slots"], s["out"], None, None, tokens, st)
    return s["out"]


def _prepare_moe_mx(c, g):
    s = _prepare_routing(c, g)
    tokens, model, inter, experts, rows = c["tokens"], c["model"], c["inter"], c["experts"], s["rows"]
    s["w1"], s["w1s"] = _quant_mx_weight(g, experts * 2 * inter, model, "fp4")
    s["w2"], s["w2s"] = _quant_mx_weight(g, experts * model, inter, "fp4")
    u8 = dict(dtype=torch.uint8, device="cuda")
    s["xq"] = torch.empty(tokens, model // 2, **u8)
    s["xs"] = torch.empty((tokens + 31) // 32 * 32, model // 32, **u8)
    s["xs_sorted"] = torch.empty((rows + 31) // 32 * 32, model // 32, **u8)
    s["hq"] = torch.empty(rows, inter // 2, **u8)
    s["hs"] = torch.empty((rows + 31) // 32 * 32, inter // 32, **u8)
    return s


def _run_moe_mx(s):
    c, st = s["case"], s["stream"]
    tokens, bm = c["tokens"], c["block"]
    _route(s, s["out"])
    if not c["inline"]:
        quant_device.per_1x32_f4_quant(s["x"], shuffle=False, stream=st, out=(s["xq"], s["xs"]))
        moe_mxfp4_sort(s["xs"][:tokens], s["sid"], s["nv"], tokens, block_size=bm, out=s["xs_sorted"], stream=st)
    kw = dict(sorted_expert_ids=s["se"], cumsum_tensor=s["nv"], BM=bm, NE=c["experts"], D_HIDDEN=c["model"], D_INTER=c["inter"], topk=c["topk"], stream=st)
    flydsl_mxfp4_gemm1(a_quant=s["xq"], a_scale_sorted_shuffled=s["xs_sorted"], w1_u8=s["w1"], w1_scale_u8=s["w1s"], m_indices=s["sid"],
                       inter_sorted_quant=s["hq"], inter_sorted_shuffled_scale=s["hs"], hidden_states=s["x"], n_tokens=tokens,
                       inline_quant=c["inline"], **kw)
    flydsl_mxfp4_gemm2(inter_sorted_quant=s["hq"], inter_sorted_shuffled_scale=s["hs"], w2_u8=s["w2"], w2_scale_u8=s["w2s"], sorted_token_ids=s["sid"],
                       sorted_weights=s["swt"], flat_out=s["out"], M_logical=tokens, max_sorted=s["rows"], epilog="atomic", **kw)
    return s["out"]


_PREPARE = {"gemm": _prepare_gemm, "mx": _prepare_mx, "moe": _prepare_moe, "moe_mx": _prepare_moe_mx}
_RUN = {"gemm": _run_gemm, "mx": _run_mx, "moe": _run_moe, "moe_mx": _run_moe_mx}


def prepare(case, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return _PREPARE[case["kind"]](case, g)


def run(state):
    return _RUN[state["case"]["kind"]](state)


def _experts_hit(c):
    """Experts that at least one token is routed to, on average over routings."""
    return c["experts"] * (1.0 - (1.0 - min(1.0, c["topk"] / c["experts"])) ** c["tokens"])


def work(case):
    c = case
    if c["kind"] == "gemm":
        m, n, k = c["M"], c["N"], c["K"]
        eb = 2 if c["dtype"] in ("bf16", "fp16") else 1
        a = m * k * 2 if eb == 2 or c["quantize"] else m * k + 4 * m
        return {"bytes": a + n * k * eb + (4 * n if eb == 1 else 0) + (2 * n if c["epilogue"] != "none" else 0) + 2 * m * n, "flops": 2.0 * m * n * k}
    if c["kind"] == "mx":
        m, n, k = c["M"], c["N"], c["K"]
        size = {"fp4": 0.5, "fp6": 0.75, "fp8": 1.0}
        a = 2 * m * k if c["quantize"] else m * k * size[c["a"]] + m * k / 32
        return {"bytes": c["batch"] * (a + n * k * size[c["b"]] + n * k / 32 + 2 * m * n), "flops": 2.0 * c["batch"] * m * n * k}
    tokens, model, inter = c["tokens"], c["model"], c["inter"]
    per_weight = (0.5 + 1.0 / 32) if c["kind"] == "moe_mx" else 0.5 if c["dtype"] == "int4" else 1.0
    scales = 0 if c["kind"] == "moe_mx" else 4 * (2 * inter + model)
    weights = _experts_hit(c) * (3 * model * inter * per_weight + scales)
    return {"bytes": weights + 4 * tokens * model + 2 * tokens * c["experts"], "flops": 6.0 * tokens * c["topk"] * model * inter}


def tolerance(case):
    c = case
    if c["kind"] in ("moe", "moe_mx"):
        # 16-bit additions of up to topk rows in arrival order, behind an intermediate that is rounded to 16 bits and quantised
        return {"rel": 1e-2, "max": 0.1}
    # fp32 (or exact int32) sums, rounded once to the output type: half a unit in the last place, now and then on the other side
    if c["out"] == "fp16":
        return {"rel": 1e-3, "max": 5e-3}
    return {"rel": 4e-3, "max": 2e-2}
