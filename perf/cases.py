"""The work that a user of this package has it do, as cases that can be timed and compared.

Every case goes through the public classes (``duqlinear4bitcuda_amd.nn``, ``duqlinear4bitcuda_amd.tools.graphs``) the
way a model's code calls them: a quantizer module and the 4-bit layers behind it, the layers with a quantizer of their
own, the 8-bit layer, the batched products of quantized attention, a stack of layers replayed as one graph, and the
conversion of a ``torch.nn.Linear``.  Sizes are those of the Llama-2 layers that the benchmark and the tests use
(4096 / 11008, 5120 / 13824, 8192 / 28672) and generic ones between them; ``draw`` covers what lies around them.

Kinds of case and their keys:

``linear4``  a 4-bit layer: ``layer``, ``tokens``, ``inf`` (a multiple of 64), ``outf``, ``bias``, ``fp6`` (the layer
             holds its 6-bit float shadow and the quantizer delivers one), ``fan`` (layers fed by one quantizer)
``linear8``  the 8-bit asymmetric layer on float32 activations: ``tokens``, ``inf`` (a multiple of 32), ``outf``, ``bias``
``matmul``   SymQuantMatMul / AsymQuantMatMul: ``sym``, ``heads``, ``rows_a``, ``rows_b``, ``width`` (a multiple of 64)
``stack``    ``layers`` quantizer + layer pairs of ``width`` x ``width``, recorded once and replayed: ``tokens``
``convert``  ``from_float`` / ``from_linear`` of a layer that lives on the GPU, and the move of the result there:
             ``layer``, ``inf``, ``outf``, ``bias``
"""
import math

import torch

from duqlinear4bitcuda_amd import nn as qnn
from duqlinear4bitcuda_amd.tools.graphs import GraphedForward

DEVICE = "cuda"
SYMMETRIC = ("Linear4bitSQ", "Linear4bitDUSQ")            # take what a SymQuantizer delivers
ASYMMETRIC = ("Linear4bitASQ", "LinearQuant4bitDUASQ", "Linear4bitASQRowSum", "LinearQuant4bitDUASQRowSum")
EIGHT_BIT = "LinearQuant8bitASQ"
DUAL_COLUMNS = 10                                         # input columns of the dual layers' first range


def listed():
    return [
        # one token of a chat through one attention projection, module calls without a graph: the smallest step there is
        {"name": "decode_1", "kind": "linear4", "layer": "Linear4bitSQ", "tokens": 1, "inf": 4096, "outf": 4096,
         "bias": False, "fp6": False, "fan": 1},
        # a batch of sixteen sequences, one token each, through the up projection of the layer with the exact zero-point correction
        {"name": "decode_16_rowsum", "kind": "linear4", "layer": "Linear4bitASQRowSum", "tokens": 16, "inf": 4096,
         "outf": 11008, "bias": True, "fp6": False, "fan": 1},
        # a serving loop's decode step: eight projections in a row, recorded once and replayed per token
        {"name": "decode_stack", "kind": "stack", "layers": 8, "tokens": 1, "width": 4096},
        # a short prompt of odd length: gate and up projection of a 13B model behind one quantizer, dual-uniform weights
        {"name": "prompt_77_gate_up", "kind": "linear4", "layer": "Linear4bitDUSQ", "tokens": 77, "inf": 5120,
         "outf": 13824, "bias": False, "fp6": False, "fan": 2},
        # the asymmetric layer on a prompt of medium length (the benchmark's fourth configuration)
        {"name": "prompt_512_asym", "kind": "linear4", "layer": "Linear4bitASQ", "tokens": 512, "inf": 4096,
         "outf": 4096, "bias": False, "fp6": False, "fan": 1},
        # prefill of 2048 tokens, the metric's own configuration, on the 6-bit float matrix path
        {"name": "prefill_2048_fp6", "kind": "linear4", "layer": "Linear4bitSQ", "tokens": 2048, "inf": 4096,
         "outf": 4096, "bias": False, "fp6": True, "fan": 1},
        # prefill as the modules run it by default (integer matrix path), a prompt that fills no tile evenly
        {"name": "prefill_1999_mlp", "kind": "linear4", "layer": "Linear4bitSQ", "tokens": 1999, "inf": 4096,
         "outf": 11008, "bias": True, "fp6": False, "fan": 1},
        # the largest layer: a 70B model's up projection, unsharded, 4096 tokens
        {"name": "prefill_4096_70b", "kind": "linear4", "layer": "Linear4bitSQ", "tokens": 4096, "inf": 8192,
         "outf": 28672, "bias": False, "fp6": True, "fan": 1},
        # decode and prefill of the 8-bit layer
        {"name": "int8_decode_8", "kind": "linear8", "tokens": 8, "inf": 4096, "outf": 4096, "bias": False},
        {"name": "int8_prefill_2048", "kind": "linear8", "tokens": 2048, "inf": 4096, "outf": 11008, "bias": True},
        # attention scores of 32 heads, 2048 queries against 2048 keys
        {"name": "attention_scores", "kind": "matmul", "sym": False, "heads": 32, "rows_a": 2048, "rows_b": 2048, "width": 128},
        # quantizing a checkpoint, one projection of it
        {"name": "convert_asym", "kind": "convert", "layer": "Linear4bitASQ", "inf": 4096, "outf": 4096, "bias": True},
    ]


def _log_uniform(rng, lo, hi, step=1):
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return int(min(hi, max(lo, round(v / step) * step)))


def draw(rng):
    kind = rng.choices(("linear4", "linear8", "matmul", "stack", "convert"), (10, 3, 3, 2, 2))[0]
    bias = rng.random() < 0.5
    if kind == "linear4":
        layer = rng.choice(SYMMETRIC + SYMMETRIC + ASYMMETRIC)   # the symmetric layers as often as the others together
        tokens = _log_uniform(rng, 1, 4096)
        fp6 = tokens > 64 and rng.random() < 0.5
        inf = _log_uniform(rng, 512, 28672, 128 if fp6 else 64)
        outf = _log_uniform(rng, 256, 28672, 16 if fp6 else 1)
        fan = rng.choice((1, 1, 2, 3)) if layer in SYMMETRIC else 1
        most = 4096 * 8192 * 28672 // (1 if fp6 else 2)          # (the integer matrix path takes longer)
        while tokens * inf * outf * fan > most:
            if fan > 1:
                fan -= 1
            else:
                tokens = max(65, tokens * 2 // 3)
        return {"kind": kind, "layer": layer, "tokens": tokens, "inf": inf, "outf": outf, "bias": bias, "fp6": fp6, "fan": fan}
    if kind == "linear8":
        return {"kind": kind, "tokens": _log_uniform(rng, 1, 2048), "inf": _log_uniform(rng, 512, 11008, 32),
                "outf": _log_uniform(rng, 256, 11008), "bias": bias}
    if kind == "matmul":
        heads, context = rng.choice((1, 8, 12, 32, 40)), _log_uniform(rng, 64, 4096, 64)
        queries = rng.choice((1, context - rng.randint(0, 9)))   # one new token per head, or a whole prompt
        dim = rng.choice((64, 128, 256))
        while heads * queries * context > 32 * 2048 * 2048:
            heads = max(1, heads // 2)
        scores = rng.random() < 0.5                               # Q K^T, or the probabilities against V
        return {"kind": kind, "sym": rng.random() < 0.5, "heads": heads, "rows_a": queries,
                "rows_b": context if scores else dim, "width": dim if scores else context}
    if kind == "stack":
        return {"kind": kind, "layers": rng.randint(2, 8), "tokens": _log_uniform(rng, 1, 64), "width": _log_uniform(rng, 1024, 8192, 64)}
    return {"kind": kind, "layer": rng.choice(SYMMETRIC + ASYMMETRIC + (EIGHT_BIT,)), "inf": _log_uniform(rng, 512, 8192, 64),
            "outf": _log_uniform(rng, 256, 8192, 16), "bias": bias}


# ---- inputs -------------------------------------------------------------------------------


def _activations(gen, rows, cols, positive=False):
    """Rows of a normalised residual stream: N(0, 1) with one channel in a hundred ten times as large; ``positive``:
    U[0, 6], what an asymmetric quantizer is for."""
    if positive:
        return torch.rand(1, rows, cols, generator=gen, device=DEVICE) * 6
    x = torch.randn(1, rows, cols, generator=gen, device=DEVICE)
    loud = torch.randint(0, cols, (max(1, cols // 100),), generator=gen, device=DEVICE)
    x[..., loud] *= 10
    return x


def _linear(gen, inf, outf, bias, dtype=torch.float16):
    """The layer of a checkpoint: weights N(0, 0.02)."""
    lin = torch.nn.Linear(inf, outf, bias=bias, device="meta", dtype=dtype)
    lin.weight = torch.nn.Parameter(torch.randn(outf, inf, generator=gen, device=DEVICE, dtype=dtype) * 0.02, requires_grad=False)
    if bias:
        lin.bias = torch.nn.Parameter(torch.randn(outf, generator=gen, device=DEVICE, dtype=dtype), requires_grad=False)
    return lin


def _scales(layer, lin):
    """The arguments that ``from_float`` of the symmetric layers takes besides the module: per-row max|W| / 7."""
    w = lin.weight.abs()
    if layer == "Linear4bitSQ":
        return (w.amax(-1, keepdim=True) / 7,)
    return w[:, :DUAL_COLUMNS].amax(-1, keepdim=True) / 7, w[:, DUAL_COLUMNS:].amax(-1, keepdim=True) / 7


def _quantized(layer, lin):
    cls = getattr(qnn, layer)
    with torch.device(DEVICE):
        new = cls.from_float(lin, *_scales(layer, lin)) if layer in SYMMETRIC else cls.from_linear(lin)
    return new.to(DEVICE)


def prepare(case, seed):
    gen = torch.Generator(device=DEVICE)
    gen.manual_seed(seed)
    kind = case["kind"]
    state = {"kind": kind}
    if kind == "linear4":
        layer = case["layer"]
        state["layers"] = [_quantized(layer, _linear(gen, case["inf"], case["outf"], case["bias"])) for _ in range(case["fan"])]
        if case["fp6"]:
            for m in state["layers"]:
                m.enable_fp6()
        if layer in SYMMETRIC:
            quantizer = qnn.SymQuantizer(shadow="only" if case["fp6"] else False)
            if case["fan"] == 1:
                state["model"] = torch.nn.Sequential(quantizer, state["layers"][0])
            else:
                state["quantizer"] = quantizer
        else:
            state["model"] = state["layers"][0]
        state["x"] = _activations(gen, case["tokens"], case["inf"], layer in ASYMMETRIC).half()
    elif kind == "linear8":
        state["model"] = _quantized(EIGHT_BIT, _linear(gen, case["inf"], case["outf"], case["bias"], torch.float32))
        state["x"] = _activations(gen, case["tokens"], case["inf"])
    elif kind == "matmul":
        shape = (1, case["heads"], case["rows_a"], case["width"])
        a = torch.randn(shape, generator=gen, device=DEVICE)
        state["a"] = (a if case["width"] <= 256 else torch.softmax(2 * a, -1)).half()
        state["b"] = torch.randn(1, case["heads"], case["rows_b"], case["width"], generator=gen, device=DEVICE).half()
        state["model"] = qnn.SymQuantMatMul() if case["sym"] else qnn.AsymQuantMatMul()
    elif kind == "stack":
        width, mods = case["width"], []
        for _ in range(case["layers"]):
            mods += [qnn.SymQuantizer(), _quantized("Linear4bitSQ", _linear(gen, width, width, False))]
        state["x"] = _activations(gen, case["tokens"], width).half()
        state["model"] = GraphedForward(torch.nn.Sequential(*mods), state["x"])
    else:
        eight = case["layer"] == EIGHT_BIT
        lin = _linear(gen, case["inf"], case["outf"], case["bias"], torch.float32 if eight else torch.float16)
        state["source"], state["layer"] = lin, case["layer"]
        state["scales"] = _scales(case["layer"], lin) if case["layer"] in SYMMETRIC else ()
    return state


def run(state):
    kind = state["kind"]
    if kind == "matmul":
        return state["model"](state["a"], state["b"])
    if kind == "convert":
        cls = getattr(qnn, state["layer"])
        make = cls.from_float if state["layer"] in SYMMETRIC else cls.from_linear
        return dict(make(state["source"], *state["scales"]).to(DEVICE).state_dict())
    if "quantizer" in state:
        x = state["quantizer"](state["x"])
        return [layer(x) for layer in state["layers"]]
    return state["model"](state["x"])


# ---- what a pass cannot do without ---------------------------------------------------------


def _channel_bytes(layer, bias):
    """Per-output-channel parameters of a layer: binary16 scales and zeros, int32 row sums, bias."""
    pairs = 2 if "DU" in layer else 1
    n = pairs * (2 if layer in SYMMETRIC else 4) + (pairs * 4 if layer.endswith("RowSum") else 0)
    if layer == EIGHT_BIT:
        return 8 + (4 if bias else 0)
    return n + (2 if bias else 0)


def work(case):
    kind = case["kind"]
    if kind == "linear4":
        t, k, n, fan = case["tokens"], case["inf"], case["outf"], case["fan"]
        return {"bytes": 2 * t * k + fan * (n * k // 2 + n * _channel_bytes(case["layer"], case["bias"]) + 2 * t * n),
                "flops": 2 * t * k * n * fan}
    if kind == "linear8":
        t, k, n = case["tokens"], case["inf"], case["outf"]
        return {"bytes": 4 * t * k + n * k + n * _channel_bytes(EIGHT_BIT, case["bias"]) + 4 * t * n, "flops": 2 * t * k * n}
    if kind == "matmul":
        h, a, b, w = case["heads"], case["rows_a"], case["rows_b"], case["width"]
        return {"bytes": 2 * h * ((a + b) * w + a * b), "flops": 2 * h * a * b * w}
    if kind == "stack":
        t, w = case["tokens"], case["width"]
        return {"bytes": case["layers"] * (w * w // 2 + 2 * w) + 4 * t * w, "flops": case["layers"] * 2 * t * w * w}
    k, n, eight = case["inf"], case["outf"], case["layer"] == EIGHT_BIT
    return {"bytes": (5 * k * n if eight else 2 * k * n + k * n // 2) + n * _channel_bytes(case["layer"], case["bias"]),
            "flops": 4 * k * n}


def tolerance(case):
    """Every path of the package gives the same bits: the accumulation is exact (integers, or floats that hold them)
    and the epilogues round once per operator in a fixed order."""
    return "exact"
