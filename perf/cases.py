"""The work that users of this package have it do, as cases with inputs, one pass and a yardstick.

A model that is served with this package calls it in three ways, and each case is one of them:

* ``w4_linear`` / ``w4_step``: linear layers with GPTQ or AWQ weights, built and loaded as a checkpoint is and then called
  as ``layer(x)`` -- one layer, or the four projections of some decoder blocks one after another (each with weights of its
  own, as a decode step walks through a model: at four blocks and more they no longer fit the caches);
* ``fp8_linear`` / ``fp8_step``: the same with FP8 weights and activations that are quantised in the call;
* ``fp8_chain``: the same block through the fused operators: RMSNorm (with the residual) + quantisation, GEMM, SiLU-mul +
  quantisation, GEMM, as a compiled model calls them;
* ``repack``: the conversion of a checkpoint's weight when it is loaded.

Sizes are those of the repository's benchmark and tests, or generic; token counts run from a single decode token over
decode batches and ragged prefill chunks to full prefill batches.
"""
from __future__ import annotations

import torch

from vllm_amd import _custom_ops as ops
from vllm_amd.layers.linear import LinearBase
from vllm_amd.layers.quantization import get_quantization_config

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}
MOST_FLOPS = 1.2e12      # of a drawn case; the largest listed one has 1.8e12


# ------------------------------------------------------------------------------------------------------------- the cases

def listed():
    big = dict(hidden=4096, kv=1024, ffn=14336)
    return [
        # one small layer, one token: what a call costs when there is hardly any work in it
        dict(name="w4 one small layer, 1 token", kind="w4_linear", form="gptq", k=2048, n=2048, tokens=1, bits=4, group=128,
             act_order=False, bias=False, dtype="bf16"),
        # single-stream decoding: every projection of eight blocks at one token, weights from memory
        dict(name="w4 decode step, 1 token", kind="w4_step", form="gptq", blocks=8, tokens=1, bits=4, group=128,
             act_order=False, bias=False, dtype="bf16", **big),
        # a served decode batch
        dict(name="w4 decode step, 32 tokens", kind="w4_step", form="gptq", blocks=4, tokens=32, bits=4, group=128,
             act_order=False, bias=False, dtype="bf16", **big),
        # an AWQ model in half precision with a few sequences
        dict(name="awq layer, 5 tokens", kind="w4_linear", form="awq", k=3584, n=18944, tokens=5, bits=4, group=128,
             act_order=False, bias=False, dtype="fp16"),
        # 8-bit GPTQ, an odd batch, with bias (a qkv projection)
        dict(name="8-bit gptq layer, 51 tokens", kind="w4_linear", form="gptq", k=3584, n=4608, tokens=51, bits=8, group=128,
             act_order=False, bias=True, dtype="fp16"),
        # a ragged prefill chunk through a layer that was quantised with act_order (rows in any order)
        dict(name="w4 desc_act layer, 333 tokens", kind="w4_linear", form="gptq", k=4096, n=6144, tokens=333, bits=4,
             group=128, act_order=True, bias=False, dtype="bf16"),
        # a full prefill batch through one block
        dict(name="awq prefill, 4096 tokens", kind="w4_step", form="awq", blocks=1, tokens=4096, bits=4, group=128,
             act_order=False, bias=False, dtype="bf16", **big),
        # FP8 decode batch, activations quantised per token in the layer
        dict(name="fp8 decode step, 16 tokens", kind="fp8_step", scheme="per_token", blocks=4, tokens=16, bias=True,
             dtype="bf16", **big),
        # a serialised FP8 checkpoint with static scales, a ragged prefill chunk
        dict(name="fp8 static layer, 250 tokens", kind="fp8_linear", scheme="static", k=5120, n=13824, tokens=250, bias=False,
             dtype="fp16"),
        # the fused operators of a block: a few tokens, then a prefill batch
        dict(name="fp8 fused block, 7 tokens", kind="fp8_chain", tokens=7, dtype="bf16", **big),
        dict(name="fp8 fused block, 2048 tokens", kind="fp8_chain", tokens=2048, dtype="bf16", **big),
        # loading a checkpoint: a gate/up projection with act_order
        dict(name="repack of a large layer", kind="repack", form="gptq", k=4096, n=28672, bits=4, act_order=True),
    ]


def _log(rng, low, high, step=1):
    """A multiple of `step` between `low` and `high`, even over their logarithm."""
    v = low * (high / low) ** rng.random()
    return int(min(high, max(low, round(v / step) * step)))


def draw(rng):
    kind = rng.choice(["w4_linear"] * 6 + ["w4_step"] * 4 + ["fp8_linear"] * 4 + ["fp8_step"] * 2 + ["fp8_chain"] * 3 + ["repack"])
    dtype = rng.choice(["bf16", "bf16", "fp16"])
    step = 128 if kind.startswith("w4") or kind == "repack" else 16
    k, n = _log(rng, 1024, 14336, step), _log(rng, 1024, 28672, 64)
    hidden = _log(rng, 1024, 6144, 128)
    block = dict(hidden=hidden, kv=rng.choice([hidden, max(128, hidden // 4 // 128 * 128)]), ffn=_log(rng, 2 * hidden, 4 * hidden, 128))
    w4 = dict(form=rng.choice(["gptq", "gptq", "awq"]), bits=4, group=rng.choice([128, 128, 128, 64, 32, -1]), act_order=False,
              bias=rng.random() < 0.3, dtype=dtype)
    if w4["form"] == "gptq":
        w4["bits"] = rng.choice([4, 4, 4, 8])
        w4["act_order"] = w4["group"] != -1 and rng.random() < 0.25
    if kind == "repack":
        return dict(kind=kind, form=w4["form"], k=k, n=n, bits=w4["bits"], act_order=w4["act_order"])
    if kind == "w4_linear":
        case = dict(kind=kind, k=k, n=n, **w4)
    elif kind == "w4_step":
        case = dict(kind=kind, blocks=rng.randint(1, 4), **w4, **block)
    elif kind == "fp8_linear":
        case = dict(kind=kind, scheme=rng.choice(["per_token", "static"]), k=k, n=n, bias=rng.random() < 0.3, dtype=dtype)
    elif kind == "fp8_step":
        case = dict(kind=kind, scheme="per_token", blocks=rng.randint(1, 4), bias=rng.random() < 0.3, dtype=dtype, **block)
    else:
        case = dict(kind=kind, dtype=dtype, **block)
    weights = sum(k * n for k, n in _shapes(case))
    most = int(MOST_FLOPS / (2 * weights))
    case["tokens"] = _log(rng, 1, max(1, min(8192 if case.get("blocks", 1) == 1 else 256, most)))
    return case


def _shapes(case):
    """(K, N) of every projection of one pass, in the order of the calls."""
    if "hidden" not in case:
        return [(case["k"], case["n"])]
    h, kv, ffn = case["hidden"], case["kv"], case["ffn"]
    return [(h, h + 2 * kv), (h, h), (h, 2 * ffn), (ffn, h)] * case.get("blocks", 1)


# ------------------------------------------------------------------------------------------------ what a program has ready

def _ints(shape, gen):
    return torch.randint(-2 ** 31, 2 ** 31 - 1, shape, dtype=torch.int32, device="cuda", generator=gen)     # uniform codes


def _randn(shape, gen, dtype, scale=1.0):
    return (torch.randn(shape, device="cuda", generator=gen) * scale).to(dtype)


def _layer(config, k, n, case, dtype):
    with torch.device("cuda"):
        return LinearBase(k, n, bias=case["bias"], quant_config=config, params_dtype=dtype, return_bias=False)


def _w4_layer(case, k, n, gen):
    dtype, group = DTYPES[case["dtype"]], case["group"]
    if case["form"] == "awq":
        config = get_quantization_config("awq_marlin").from_config(dict(bits=4, group_size=group, zero_point=True))
    else:
        config = get_quantization_config("gptq_marlin").from_config(
            dict(bits=case["bits"], group_size=group, desc_act=case["act_order"], sym=True))
    layer = _layer(config, k, n, case, dtype)
    layer.qweight.data = _ints(layer.qweight.shape, gen)
    layer.scales.data = ((torch.randn(layer.scales.shape, device="cuda", generator=gen).abs() * 0.01 + 1e-3)
                         * (1.0 if case["bits"] == 4 else 1 / 16)).to(dtype)
    layer.qzeros.data = _ints(layer.qzeros.shape, gen)
    if case["form"] == "gptq":
        rows = torch.arange(k, dtype=torch.int32, device="cuda")
        if case["act_order"]:
            rows = rows[torch.randperm(k, device="cuda", generator=gen)]
        layer.g_idx.data = (rows // (group if group > 0 else k)).contiguous()
    if case["bias"]:
        layer.bias.data = _randn((n,), gen, dtype, 0.01)
    layer.process_weights_after_loading()
    return layer


def _fp8_layer(case, k, n, gen):
    dtype = DTYPES[case["dtype"]]
    if case["scheme"] == "static":
        config = get_quantization_config("fp8").from_config(dict(quant_method="fp8", activation_scheme="static"))
    else:
        config = get_quantization_config("ptpc_fp8").from_config({})
    layer = _layer(config, k, n, case, dtype)
    w = _randn((n, k), gen, dtype, 0.02)
    if case["scheme"] == "static":
        layer.weight.data, scale = ops.scaled_fp8_quant(w)
        layer.weight_scale.data = scale.reshape(1)
        layer.input_scale.data = torch.full((1,), 5.0 / 448, device="cuda")
    else:
        layer.weight.data = w
    if case["bias"]:
        layer.bias.data = _randn((n,), gen, dtype, 0.01)
    layer.process_weights_after_loading()
    return layer


def _chain(case, gen):
    dtype, m, h, ffn = DTYPES[case["dtype"]], case["tokens"], case["hidden"], case["ffn"]
    weights = []
    for k, n in _shapes(case):
        q, s = ops.scaled_fp8_quant(_randn((n, k), gen, dtype, 0.02), use_per_token_if_dynamic=True)
        weights.append((q.t(), s))
    return dict(x=_randn((m, h), gen, dtype), attn=_randn((m, h), gen, dtype), residual=_randn((m, h), gen, dtype),
                norms=[_randn((h,), gen, dtype, 0.1) + 1 for _ in range(2)], weights=weights, dtype=dtype,
                act=torch.empty((m, ffn), dtype=ops.FP8_DTYPE, device="cuda"), act_scale=torch.full((1,), 4.0 / 448, device="cuda"))


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    kind = case["kind"]
    if kind == "repack":
        k, n, bits = case["k"], case["n"], case["bits"]
        shape = (k, n * bits // 32) if case["form"] == "awq" else (k * bits // 32, n)
        perm = torch.randperm(k, device="cuda", generator=gen).int() if case["act_order"] else torch.empty(0, dtype=torch.int32, device="cuda")
        return dict(kind=kind, form=case["form"], codes=_ints(shape, gen), perm=perm, k=k, n=n, bits=bits)
    if kind == "fp8_chain":
        return dict(kind=kind, **_chain(case, gen))
    make = _w4_layer if kind.startswith("w4") else _fp8_layer
    dtype = DTYPES[case["dtype"]]
    return dict(kind=kind, calls=[(make(case, k, n, gen), _randn((case["tokens"], k), gen, dtype)) for k, n in _shapes(case)])


# -------------------------------------------------------------------------------------------------------------- one pass

def _run_chain(s):
    (wqkv, sqkv), (wo, so), (wgu, sgu), (wd, sd) = s["weights"]
    dtype = s["dtype"]
    q, qs = ops.rms_norm_dynamic_per_token_quant(s["x"], s["norms"][0], 1e-5, ops.FP8_DTYPE, residual=s["residual"])
    qkv = ops.cutlass_scaled_mm(q, wqkv, qs, sqkv, dtype)
    q, qs = ops.scaled_fp8_quant(s["attn"], use_per_token_if_dynamic=True)
    o = ops.cutlass_scaled_mm(q, wo, qs, so, dtype)
    q, qs = ops.rms_norm_dynamic_per_token_quant(o, s["norms"][1], 1e-5, ops.FP8_DTYPE, residual=s["residual"])
    gate_up = ops.cutlass_scaled_mm(q, wgu, qs, sgu, dtype)
    ops.silu_and_mul_quant(s["act"], gate_up, s["act_scale"])
    down = ops.cutlass_scaled_mm(s["act"], wd, s["act_scale"], sd, dtype)
    return [qkv, o, gate_up, down, s["residual"]]


def run(state):
    kind = state["kind"]
    if kind == "repack":
        if state["form"] == "awq":
            return ops.awq_marlin_repack(state["codes"], state["k"], state["n"], state["bits"])
        return ops.gptq_marlin_repack(state["codes"], state["perm"], state["k"], state["n"], state["bits"])
    if kind == "fp8_chain":
        return _run_chain(state)
    return [layer(x) for layer, x in state["calls"]]


# ------------------------------------------------------------------------------------------------------------ yardsticks

def work(case):
    kind = case["kind"]
    if kind == "repack":
        return {"bytes": 2 * case["k"] * case["n"] * case["bits"] // 8 + (4 * case["k"] if case["act_order"] else 0), "flops": 0}
    m, total, flops = case["tokens"], 0, 0
    for k, n in _shapes(case):
        flops += 2 * m * n * k
        total += 2 * m * k + 2 * m * n + (2 * n if case.get("bias") else 0)
        if kind.startswith("w4"):
            groups = k // case["group"] if case["group"] > 0 else 1
            total += k * n * case["bits"] // 8 + groups * n * 2 + (groups * n // 2 if case["form"] == "awq" else 0)
            total += 4 * k if case["act_order"] else 0
        else:
            total += k * n + 4 * n
    if kind == "fp8_chain":
        total += 4 * m * case["hidden"] + 4 * case["hidden"]      # the residual in and out, the norms' weights
    return {"bytes": total, "flops": flops}


def tolerance(case):
    """Whole words of a repacked weight are what they are.  A GEMM's output is rounded to 16 bits once (2^-9 or 2^-12 of the value)
    and may take its weights rounded to 16 bits or not; a sum of squares in another order moves an FP8 code of a normalised
    activation (a step of 1/16) now and then."""
    if case["kind"] == "repack":
        return "exact"
    if case["kind"] == "fp8_chain":
        return {"rel": 8e-3}
    return {"rel": 5e-3} if case["dtype"] == "bf16" else {"rel": 1e-3}
