"""The work that users of this package have it do, as timed cases.

The package is one operator and the modules around it: ``cascaded_lowp_matmul`` called directly on two
tensors, ``BasedXLLowPLinear`` in the place of every ``nn.Linear`` of a UNet, ``BasedXLFusedKV`` /
``BasedXLFusedQKV`` for attention projections, and ``BasedXLLowPGEGLU`` followed by a Linear for
feed-forward blocks.  It runs forward only.  Activations are N(0, 1), weights N(0, 0.02) (N(0, 1) for the
square products of the operator's own benchmark), as in ``bench.py`` and ``unet_shapes.py``.

A case is ``{kind, dtype, lowp, terms, prepared, m, k, n}``: ``m`` rows of activations, ``k`` input features,
``n`` output features (for ``ffn``: k -> 2 n gated -> n -> k).  ``lowp`` "" takes the operator's default
cascade for the dtype: two bf16 terms for fp32 tensors, one term of their own format for fp16 / bf16.
"""
import math

import torch
import torch.nn as nn

from basedxl_amd import cascaded_lowp_matmul
from basedxl_amd.modules.fused_kv import BasedXLFusedKV, BasedXLFusedQKV
from basedxl_amd.modules.geglu import BasedXLLowPGEGLU
from basedxl_amd.modules.lowp_linear import BasedXLLowPLinear

_DTYPES = {"fp32": torch.float32, "fp16": torch.float16, "bf16": torch.bfloat16}


def _case(kind, m, k, n, *, dtype="fp32", lowp="", terms=0, prepared=False, name=None):
    c = {"kind": kind, "dtype": dtype, "lowp": lowp, "terms": terms, "prepared": prepared, "m": m, "k": k, "n": n}
    return c if name is None else {"name": name, **c}


def listed():
    return [
        # time / size embedding layers: two rows (the guided batch), some twenty calls per UNet step, latency only
        _case("linear", 2, 1280, 1280, name="embedding_fp32"),
        # keys and values of the 2 x 77 text tokens in one projection: skinny, weights read once
        _case("kv", 154, 2048, 1280, name="text_kv_fp32"),
        # an attention projection of the 64 x 64 stage on half a latent, the operator called on raw tensors
        _case("matmul", 4096, 640, 640, name="attention_proj_fp32"),
        # query / key / value of the 32 x 32 stage, weights kept split; the rows of an 832 x 1216 image
        # (2 x 26 x 38 tokens), as every aspect ratio but the square one has row counts off the tile sizes
        _case("qkv", 1976, 1280, 1280, prepared=True, name="qkv_bucket_fp32"),
        # the feed-forward block of the 32 x 32 stage (the benchmark's shape), weights split in every call
        _case("ffn", 2048, 1280, 5120, name="ffn_fp32"),
        # the most frequent layer of a UNet step in the dtype that the reference runs its UNet in
        _case("linear", 2048, 1280, 1280, dtype="fp16", prepared=True, name="linear_fp16"),
        # the feed-forward block in that dtype
        _case("ffn", 2048, 1280, 5120, dtype="fp16", prepared=True, name="ffn_fp16"),
        # the square sweep that the operator is benchmarked with, near its upper end and in its middle
        _case("matmul", 4096, 4096, 4096, name="square_fp32"),
        _case("matmul", 2048, 2048, 2048, dtype="fp16", name="square_fp16"),
        # the other cascades that are run on a UNet: three fp8 terms (the activations' scale found in every
        # call) and, where fp32 accuracy is wanted, three fp16 terms
        _case("linear", 2048, 1280, 1280, lowp="fp8", terms=3, prepared=True, name="linear_fp8x3"),
        _case("matmul", 2048, 1280, 10240, lowp="fp16", terms=3, name="ffn_up_fp16x3"),
        # no dimension a multiple of anything (the ragged shape of the accuracy tests)
        _case("matmul", 333, 456, 211, name="ragged_fp32"),
    ]


#: multiply-adds x products of the largest listed case: no drawn one has more
_MOST = 3 * 4096 ** 3


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _features(rng, lo, hi):
    """Layer widths: mostly multiples of 64, some of 8, some anything."""
    x, r = _log(rng, lo, hi), rng.random()
    unit = 64 if r < 0.65 else 8 if r < 0.85 else 1
    return max(unit, (x + unit // 2) // unit * unit)


def _rows(rng, lo, hi):
    """Token counts: half of them whole multiples of 64, the others as image sizes and prompts give them."""
    x = _log(rng, lo, hi)
    return max(1, (x + 32) // 64 * 64) if x >= 64 and rng.random() < 0.5 else x


def draw(rng):
    kind = rng.choice(("linear", "linear", "matmul", "matmul", "kv", "qkv", "ffn", "square"))
    cascade = rng.choice((("fp32", "", 0),) * 4 + (("fp16", "", 0),) * 2 + (("bf16", "", 0), ("fp32", "fp8", 3), ("fp32", "fp16", 3)))
    if kind in ("ffn", "kv", "qkv") and cascade[1]:
        cascade = ("fp32", "", 0)       # (the three-term cascades: single layers and plain products)
    prepared = cascade[0] != "fp32" or rng.random() < 0.5
    if cascade[1:] == ("fp16", 3) or kind in ("matmul", "square"):
        prepared = False                # (raw tensors)
    if kind == "square":
        kind = "matmul"
        m = k = n = _features(rng, 256, 4096)
    elif kind == "kv":
        m, k, n = _rows(rng, 16, 320), _features(rng, 768, 2048), _features(rng, 320, 1280)
    elif kind == "ffn":
        m, k = _rows(rng, 64, 8192), _features(rng, 320, 1280)
        n = 4 * k
    elif kind == "qkv":
        m, k = _rows(rng, 64, 8192), _features(rng, 320, 1280)
        n = k
    else:
        m, k, n = _rows(rng, 2, 8192), _features(rng, 320, 5120), _features(rng, 320, 10240)
    case = _case(kind, m, k, n, dtype=cascade[0], lowp=cascade[1], terms=cascade[2], prepared=prepared)
    macs, most = _macs(case), (0.75 if case["terms"] == 3 else 1.0) * _MOST    # (three terms: passes over the operands besides)
    if macs > most:
        case["m"] = max(1, int(m * most / macs))
        if kind == "matmul" and m == k == n:
            case["m"] = case["k"] = case["n"] = _log(rng, 1024, 2944)          # (6 x 2944^3 < 0.75 x 3 x 4096^3)
    return case


def _products(case):
    if case["terms"] == 3:
        return 6
    return 1 if case["dtype"] != "fp32" else 3


def _macs(case):
    m, k, n = case["m"], case["k"], case["n"]
    per_row = {"linear": k * n, "matmul": k * n, "kv": 2 * k * n, "qkv": 3 * k * n, "ffn": 3 * k * n}[case["kind"]]
    return m * per_row * _products(case)


def work(case):
    m, k, n = case["m"], case["k"], case["n"]
    size = 4 if case["dtype"] == "fp32" else 2
    weights = {"linear": k * n + n, "matmul": k * n, "kv": 2 * k * n, "qkv": 3 * k * n, "ffn": 3 * k * n + 2 * n + k}[case["kind"]]
    result = {"linear": m * n, "matmul": m * n, "kv": 2 * m * n, "qkv": 3 * m * n, "ffn": m * k}[case["kind"]]
    return {"bytes": size * (m * k + weights + result), "flops": 2 * _macs(case)}


def tolerance(case):
    """Four times what the path shows against the same product in 64 bits: relative error, and largest
    difference over the result's root mean square.  Measured over the listed and drawn cases: 4.5e-6 / 2.5e-5
    for two bf16 terms, 1.5e-7 / 9.9e-7 for three fp16 terms, 3.5e-5 / 1.8e-4 for three fp8 terms, 2.1e-4 / 4.9e-4
    for fp16 and 1.7e-3 / 3.9e-3 for bf16 tensors (the rounding of the result); a feed-forward block, two products
    one after the other, shows about 1.7 times that (largest difference 2.5 times)."""
    if case["lowp"] == "fp8":
        rel, big = 1.4e-4, 7.2e-4
    elif case["lowp"] == "fp16":
        rel, big = 6.0e-7, 4.0e-6
    else:
        rel, big = {"fp32": (1.8e-5, 1.0e-4), "fp16": (8.3e-4, 2.0e-3), "bf16": (6.7e-3, 1.6e-2)}[case["dtype"]]
    return {"rel": 1.7 * rel, "max": 2.5 * big} if case["kind"] == "ffn" else {"rel": rel, "max": big}


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    dtype, kind = _DTYPES[case["dtype"]], case["kind"]
    m, k, n = case["m"], case["k"], case["n"]
    options = {"lowp": case["lowp"], "terms": case["terms"]} if case["lowp"] else {}

    def normal(*shape, std=1.0):
        return (torch.randn(*shape, device="cuda", generator=gen) * std).to(dtype)

    def layer(inputs, outputs, bias=True):
        lin = nn.Linear(inputs, outputs, bias=bias, device="meta").to_empty(device="cuda").to(dtype).requires_grad_(False)
        lin.weight.copy_(normal(outputs, inputs, std=0.02))
        if bias:
            lin.bias.copy_(normal(outputs, std=0.02))
        return lin

    state = {"kind": kind, "x": normal(m, k)}
    if kind == "matmul":
        state["w"] = normal(k, n, std=1.0 if m == k == n else 0.02)
        state["options"] = options
        return state
    options["prepared"] = case["prepared"]
    if kind == "linear":
        state["layer"] = BasedXLLowPLinear(layer(k, n), **options)
        state["layer"].prepare()
    elif kind == "kv":
        state["layer"] = BasedXLFusedKV(layer(k, n, False), layer(k, n, False), **options)
        state["layer"].to_kv.prepare()
    elif kind == "qkv":
        state["layer"] = BasedXLFusedQKV(layer(k, n, False), layer(k, n, False), layer(k, n, False), **options)
        state["layer"].to_qkv.prepare()
    else:
        state["up"] = BasedXLLowPGEGLU(layer(k, 2 * n), **options)
        state["down"] = BasedXLLowPLinear(layer(n, k), **options)
        state["up"].prepare()
        state["down"].prepare()
    return state


def run(state):
    if state["kind"] == "matmul":
        return cascaded_lowp_matmul(state["x"], state["w"], **state["options"])
    if state["kind"] == "ffn":
        return state["down"](state["up"](state["x"]))
    return state["layer"](state["x"])
