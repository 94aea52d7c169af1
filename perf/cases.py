"""The fused Matmul -> row-Softmax calls that this library's users make, as
cases to time and to compare: what goes in, one call, what comes out.

    listed()            the cases
    draw(rng)           one more case of the same ranges
    prepare(case, seed) inputs on the GPU, made from the seed alone
    run(state)          one call of ``chain.matmul_softmax``
    exact(case, seed)   the same result in 64 bits, by plain torch
    work(case)          bytes and floating-point operations a call cannot do without
    tolerance(case)     the largest relative error of a correct implementation

A case is a dict of plain values: batch (0: 2-D operands), m, n, k, the input
and output types, and the law of the inputs (see prepare).

The ranges.  General products (m, n, k from one tile to a few thousand, every
input type), attention scores in prefill (heads * sequences up to 64, head
dim up to 128) and in decode (one to eight query rows per head against a long
key cache), and wide-row logits over a vocabulary, in prefill and in decode.
Sizes are odd as often as not: m is any number, n a multiple of 8 and k of 16
bytes, which is all that the entry point asks for.
"""
from __future__ import annotations

import math

import torch

from welder_typical_chain_amd.chain import matmul_softmax

_TORCH = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16,
          "fp8": torch.float8_e4m3fn}
_BYTES = {"f32": 4, "f16": 2, "bf16": 2, "fp8": 1}
_FP8_MAX = 448.0

# No drawn case does more than the largest listed ones: 2 * 8192 * 8192 * 4096
# operations (f32, whose matrix rate is a sixteenth: 2 * 2048**3), and the
# bytes of 64 heads of 2048 x 2048 scores.
_MOST_FLOPS = 2 * 8192 * 8192 * 4096
_MOST_F32_FLOPS = 2 * 2048 ** 3
_MOST_BYTES = 600_000_000


def _case(name, batch, m, n, k, in_dtype, out_dtype, law):
    return {"name": name, "batch": batch, "m": m, "n": n, "k": k, "in_dtype": in_dtype,
            "out_dtype": out_dtype, "law": law}


def listed():
    return [
        # the smallest chain: one tile, where the launch and the host are the cost
        _case("chain_f32_128", 0, 128, 128, 128, "f32", "f32", "uniform"),
        # the tall, narrow chain that the A/B harness pins: f16 in, f32 out
        _case("tall_f16_f32", 0, 8192, 128, 64, "f16", "f32", "unit"),
        # the headline product
        _case("square_f16", 0, 2048, 2048, 1024, "f16", "f16", "flat"),
        # an ordinary product of no particular size, bf16 throughout
        _case("ragged_bf16", 0, 1500, 3000, 1000, "bf16", "bf16", "unit"),
        # an f32 product of ordinary size
        _case("square_f32", 0, 1024, 1024, 1024, "f32", "f32", "unit"),
        # an fp8 product with per-tensor scales, odd sizes
        _case("ragged_fp8", 0, 1000, 4104, 2064, "fp8", "bf16", "amax"),
        # attention scores in prefill: many heads, long sequence
        _case("attn_prefill_f16", 64, 2048, 2048, 128, "f16", "f16", "attention"),
        # attention scores in prefill: head dim 64, odd sequence lengths
        _case("attn_ragged_bf16", 24, 777, 1000, 64, "bf16", "bf16", "attention"),
        # attention scores in decode: four query rows a key head, long cache
        _case("attn_decode_f16", 128, 4, 2048, 128, "f16", "f16", "attention"),
        # vocabulary logits of one decode step of eight sequences
        _case("logits_decode_bf16", 0, 8, 32768, 4096, "bf16", "f16", "half"),
        # vocabulary logits in prefill
        _case("logits_prefill_bf16", 0, 1024, 32768, 4096, "bf16", "f16", "half"),
        # the largest product, fp8 with per-tensor scales
        _case("large_fp8", 0, 8192, 8192, 4096, "fp8", "f16", "amax"),
    ]


def _log_size(rng, lo, hi, step=1):
    """A multiple of `step` in [lo, hi], spread over its logarithm."""
    x = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(step, int(round(x / step)) * step)


def _drawn(rng):
    kind = rng.choice(["general", "general", "attn_prefill", "attn_decode", "logits_prefill",
                       "logits_decode"])
    if kind == "general":
        in_dtype = rng.choice(["f16", "bf16", "fp8", "f32"])
        out_dtype = "f32" if in_dtype == "f32" else rng.choice(["f16", "bf16", "f32"])
        hi = 4096 if in_dtype == "f32" else 8192
        return (rng.choice([0, 0, 0, 2, 4]), _log_size(rng, 64, hi), _log_size(rng, 64, hi, 8),
                _log_size(rng, 64, 4096, 16), in_dtype, out_dtype,
                "amax" if in_dtype == "fp8" else rng.choice(["unit", "flat"]))
    if kind == "attn_prefill":
        t = rng.choice(["f16", "bf16"])
        n = _log_size(rng, 128, 2048, 8)
        m = n if rng.random() < 0.5 else _log_size(rng, 64, 2048)
        return (_log_size(rng, 4, 64), m, n, rng.choice([32, 64, 80, 96, 128]), t,
                rng.choice([t, t, "f32"]), "attention")
    if kind == "attn_decode":
        t = rng.choice(["f16", "bf16"])
        return (_log_size(rng, 8, 512), rng.choice([1, 1, 2, 4, 5, 8]), _log_size(rng, 256, 8192, 8),
                rng.choice([64, 96, 128]), t, rng.choice([t, t, "f32"]), "attention")
    in_dtype = rng.choice(["f16", "bf16", "fp8"])
    m = _log_size(rng, 1, 64) if kind == "logits_decode" else _log_size(rng, 65, 1024)
    return (0, m, _log_size(rng, 8192, 65536, 8), _log_size(rng, 1024, 8192, 16), in_dtype,
            rng.choice(["f16", "bf16", "f32"]), "amax" if in_dtype == "fp8" else "half")


def draw(rng):
    while True:
        batch, m, n, k, in_dtype, out_dtype, law = _drawn(rng)
        case = {"batch": batch, "m": m, "n": n, "k": k, "in_dtype": in_dtype,
                "out_dtype": out_dtype, "law": law}
        w = work(case)
        most = _MOST_F32_FLOPS if in_dtype == "f32" else _MOST_FLOPS
        if w["flops"] <= most and w["bytes"] <= _MOST_BYTES:
            return case


def work(case):
    b, m, n, k = max(case["batch"], 1), case["m"], case["n"], case["k"]
    return {"bytes": b * ((m * k + k * n) * _BYTES[case["in_dtype"]] +
                          m * n * _BYTES[case["out_dtype"]]),
            "flops": 2 * b * m * n * k}


def _operands(case, seed):
    """a, b and the keyword scales of a case.

    The laws: "uniform" U(-1, 1) on both; "half" U(-1/2, 1/2) on both; "flat"
    N(0, 1/k) on both; "unit" a N(0, 1/k) and b N(0, 1), logits of deviation
    1; "attention" N(0, 1) on both with logit scale 1/sqrt(k); "amax" N(0, 1)
    quantised to e4m3 with one scale per tensor that takes its largest value
    to the type's largest.
    """
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    lead = (case["batch"],) if case["batch"] else ()
    m, n, k, law = case["m"], case["n"], case["k"], case["law"]
    dtype = _TORCH[case["in_dtype"]]

    def make(shape, deviation):
        if law in ("uniform", "half"):
            width = 2.0 if law == "uniform" else 1.0
            return (torch.rand(shape, generator=g, device="cuda") - 0.5) * width
        return torch.randn(shape, generator=g, device="cuda") * deviation

    root = 1.0 / math.sqrt(k)
    a = make(lead + (m, k), root if law in ("flat", "unit") else 1.0)
    b = make(lead + (k, n), root if law == "flat" else 1.0)
    scales = {}
    if law == "attention":
        scales["logit_scale"] = root
    if law == "amax":
        sa, sb = (float(x.abs().max()) / _FP8_MAX for x in (a, b))
        a, b = a / sa, b / sb
        scales.update(scale_a=sa, scale_b=sb)
    return a.to(dtype), b.to(dtype), scales


def prepare(case, seed):
    a, b, scales = _operands(case, seed)
    out = torch.empty(a.shape[:-1] + (case["n"],), dtype=_TORCH[case["out_dtype"]], device="cuda")
    return {"a": a, "b": b, "out": out, "scales": scales}


def run(state):
    return matmul_softmax(state["a"], state["b"], out=state["out"], **state["scales"])


def exact(case, seed):
    a, b, scales = _operands(case, seed)
    scale = math.prod(scales.values())
    if a.dim() == 2:
        a, b = a[None], b[None]
    out = torch.empty(a.shape[:-1] + (case["n"],), dtype=torch.float64, device="cuda")
    for i in range(a.shape[0]):  # e4m3 has no direct conversion to 64 bits
        y = torch.matmul(a[i].float().double(), b[i].float().double())
        torch.softmax(y.mul_(scale), dim=-1, out=out[i])
    return out if case["batch"] else out[0]


def tolerance(case):
    """About four times the largest error against `exact` over the ranges above:
    one rounding to the output type (f16 2.7e-4, bf16 2.0e-3; f16 values that
    a rescaling pass rounds twice are among these), and in f32 the error of
    the logits, which the exponential turns into a relative one: logits of
    deviation near 1 2e-6, of deviation 3 to 8 6e-6, the fp8 products' (of
    deviation sqrt(k), up to several hundred) 1.2e-4.  "max" is a few units in
    the last place of the output type.
    """
    if case["out_dtype"] == "f16":
        return {"rel": 1e-3, "max": 4e-3}
    if case["out_dtype"] == "bf16":
        return {"rel": 8e-3, "max": 2e-2}
    if case["law"] == "amax":
        return {"rel": 5e-4, "max": 4e-3}
    return {"rel": 2e-5 if case["law"] == "half" else 8e-6, "max": 2e-4}
