"""Performance cases: the calls that a serving program makes through the public entry points, over the range of
sizes, data types and options that it meets.

Four kinds of case, each one pass of one part of a transformer layer over packed (layout-A) weights:

  gemv    `gemv_layoutA`: one token through one linear layer (decode at batch one); bf16, fp16 or soft-FP8 weights
  linear  `gemm_layoutA_linear`: 2 to 4096 tokens through one linear layer, from a decode batch to a prefill; the
          soft-FP8 weights come with one fp32 scale per 128 x 128 block, drawn at random like a trained checkpoint's
  chain   `layoutB` -> `gemm_layoutABC` -> `gemm_layoutAB_ContinuousC`: two products whose activations stay in the
          native layout in between, 16 to 1024 tokens
  moe     `fused_moe`: router, grouped gate/up product with SiLU, down product and weighted sum; 1 to 2048 tokens,
          bf16, fp16 or soft-FP8 weights, plain softmax routing or grouped sigmoid routing with a selection bias

`rows` and `k` are those of the weight matrix, `tokens` the rows of the activations.
"""
import math

import torch

import muxi_layout_kernels as mlk
from muxi_layout_kernels.muxi_moe_planC import fused_moe

_DTYPE = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp8": torch.bfloat16}    # of the activations
_BYTES = {"bf16": 2, "fp16": 2, "fp8": 1}                                            # of a weight

# Weight shapes (rows, k) of the packaged launch-parameter tables and of the benchmark.
_SHAPES = [(4096, 4096), (11008, 4096), (4096, 11008), (12288, 4096), (22016, 4096), (32000, 4096), (8192, 8192),
           (28672, 4096), (4096, 14336), (28672, 8192), (8192, 14336), (4608, 3584), (37888, 3584), (3584, 18944),
           (4608, 7168), (3072, 1536), (7168, 2048), (512, 7168), (7168, 2304), (1280, 5120), (5120, 640), (13824, 5120),
           (5120, 13824), (10240, 8192), (27648, 5120)]
# Expert layers (experts, picks, hidden, intermediate, routing groups, kept groups): the benchmark's layer, two
# layers of the repository's tests, and two of generic sizes in between.
_MOE = [(8, 2, 4096, 14336, 1, 1), (256, 8, 7168, 256, 8, 4), (128, 8, 2048, 768, 1, 1), (16, 4, 4096, 2048, 1, 1),
        (64, 6, 2048, 1024, 1, 1)]
_MAX_FLOPS = 1.45e12     # of the largest listed case


def _gemv(name, rows, k, weights, bias=False):
    return {"name": name, "kind": "gemv", "rows": rows, "k": k, "tokens": 1, "weights": weights, "bias": bias}


def _linear(name, rows, k, tokens, weights, bias=False):
    return {"name": name, "kind": "linear", "rows": rows, "k": k, "tokens": tokens, "weights": weights, "bias": bias}


def _moe(name, layer, tokens, weights, sigmoid=False):
    e, picks, hidden, inter, groups, kept = layer
    return {"name": name, "kind": "moe", "experts": e, "picks": picks, "hidden": hidden, "inter": inter,
            "groups": groups, "kept": kept, "tokens": tokens, "weights": weights, "sigmoid": sigmoid}


def listed():
    return [
        # decode of one token through an attention projection: the smallest call, launch latency counts
        _gemv("gemv_bf16_4096x4096", 4096, 4096, "bf16"),
        # decode of one token through a large feed-forward matrix held in fp8
        _gemv("gemv_fp8_28672x8192", 28672, 8192, "fp8"),
        # a decode batch of sixteen through a feed-forward matrix: the benchmark's headline
        _linear("gemm_fp16_11008x4096_t16", 11008, 4096, 16, "fp16"),
        # an odd decode batch through a linear layer with a bias, fp8 weights
        _linear("linear_fp8_14336x8192_t33", 14336, 8192, 33, "fp8", True),
        # a decode batch through two products that hand the native layout on
        {"name": "chain_bf16_11008_t64", "kind": "chain", "rows": 11008, "k": 4096, "rows2": 4096, "tokens": 64,
         "weights": "bf16"},
        # a short prompt
        _linear("gemm_fp16_11008x4096_t300", 11008, 4096, 300, "fp16"),
        # a long prompt, ragged, with a bias, on a shape that the launch-parameter table does not hold
        _linear("gemm_bf16_13824x5120_t3000", 13824, 5120, 3000, "bf16", True),
        # a prompt through a large matrix held in fp8
        _linear("linear_fp8_28672x8192_t1024", 28672, 8192, 1024, "fp8"),
        # one token through an expert layer held in fp8
        _moe("moe_fp8_8experts_t1", _MOE[0], 1, "fp8"),
        # a decode batch through the same layer in bf16
        _moe("moe_bf16_8experts_t48", _MOE[0], 48, "bf16"),
        # a large decode batch through many small experts with grouped routing
        _moe("moe_fp8_256experts_t256", _MOE[1], 256, "fp8", True),
        # a prefill through an expert layer: the largest call
        _moe("moe_bf16_8experts_t2048", _MOE[0], 2048, "bf16"),
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _draw_shape(rng):
    """A weight shape of the tables, or one of the same range whose sides are any multiples of 128."""
    if rng.random() < 0.5:
        return rng.choice(_SHAPES)
    while True:
        rows, k = 128 * _log_int(rng, 4, 300), 128 * _log_int(rng, 4, 144)
        if rows * k <= 28672 * 8192:
            return rows, k


def draw(rng):
    kind = rng.choice(["gemv", "linear", "linear", "linear", "chain", "moe", "moe", "moe"])
    if kind == "gemv":
        rows, k = _draw_shape(rng)
        case = _gemv("", rows, k, rng.choice(["bf16", "fp16", "fp8"]), rng.random() < 0.3)
    elif kind == "linear":
        rows, k = _draw_shape(rng)
        tokens = _log_int(rng, 2, min(4096, _MAX_FLOPS / (2 * rows * k)))
        case = _linear("", rows, k, tokens, rng.choice(["bf16", "fp16", "fp8"]), rng.random() < 0.3)
    elif kind == "chain":
        rows, k = _draw_shape(rng)
        tokens = 16 * _log_int(rng, 1, 64)
        case = {"kind": "chain", "rows": rows, "k": k, "rows2": 128 * _log_int(rng, 4, 64), "tokens": tokens,
                "weights": rng.choice(["bf16", "fp16"])}
    else:
        layer = rng.choice(_MOE)
        case = _moe("", layer, _log_int(rng, 1, 2048), rng.choice(["bf16", "fp16", "fp8"]), layer[4] > 1)
    case.pop("name", None)
    return case


def _randn(gen, shape, dtype, std):
    return (torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32) * std).to(dtype)


def _weights(gen, rows, k, kind):
    """One packed weight matrix and its block scales (None for 16-bit weights): N(0, 1 / k) in all."""
    if kind != "fp8":
        return mlk.pack_layout_a(_randn(gen, (rows, k), _DTYPE[kind], k ** -0.5)), None
    codes = (torch.randn((rows, k), generator=gen, device="cuda") * 16).clamp_(-448, 448).to(torch.float8_e4m3fn)
    scale = (torch.rand(((rows + 127) // 128, (k + 127) // 128), generator=gen, device="cuda") + 0.5) * (k ** -0.5 / 16)
    return mlk.pack_layout_a(codes.view(torch.uint8)), scale


def _expert_weights(gen, experts, rows, k, kind):
    """Packed weights [experts, rows, k] and scales, made expert by expert."""
    packed = torch.empty((experts, rows, k), dtype=torch.uint8 if kind == "fp8" else _DTYPE[kind], device="cuda")
    scales = torch.empty((experts, rows // 128, k // 128), device="cuda") if kind == "fp8" else None
    for e in range(experts):
        w, s = _weights(gen, rows, k, kind)
        packed[e] = w.view(rows, k)
        if s is not None:
            scales[e] = s
    return packed, scales


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    dtype, kind = _DTYPE[case["weights"]], case["kind"]
    tokens = case["tokens"]
    state = {"kind": kind, "case": case}
    if kind in ("gemv", "linear"):
        state["w"], state["scale"] = _weights(gen, case["rows"], case["k"], case["weights"])
        state["x"] = _randn(gen, (tokens, case["k"]), dtype, 1.0)
        state["bias"] = _randn(gen, (1, case["rows"]), dtype, 1.0) if case["bias"] else None
    elif kind == "chain":
        state["w1"], _ = _weights(gen, case["rows"], case["k"], case["weights"])
        state["w2"], _ = _weights(gen, case["rows2"], case["rows"], case["weights"])
        state["x"] = _randn(gen, (tokens, case["k"]), dtype, 1.0)
    else:
        e, hidden, inter = case["experts"], case["hidden"], case["inter"]
        state["w1"], state["w1_scale"] = _expert_weights(gen, e, 2 * inter, hidden, case["weights"])
        state["w2"], state["w2_scale"] = _expert_weights(gen, e, hidden, inter, case["weights"])
        state["x"] = _randn(gen, (tokens, hidden), dtype, 1.0)
        state["logits"] = _randn(gen, (tokens, e), dtype, 1.0)
        options = {"renormalize": True, "score_func": "sigmoid" if case["sigmoid"] else "softmax"}
        if case["groups"] > 1:
            options.update(use_grouped_topk=True, num_expert_group=case["groups"], topk_group=case["kept"],
                           gating_bias=_randn(gen, (e,), dtype, 0.1))
        if case["weights"] == "fp8":
            options.update(w1_scale=state["w1_scale"], w2_scale=state["w2_scale"], block_shape=[128, 128], soft_fp8=True)
        state["options"] = options
    return state


def run(state):
    kind = state["kind"]
    if kind == "gemv":
        return mlk.gemv_layoutA(state["w"], state["x"], scale_matrix=state["scale"], bias=state["bias"])
    if kind == "linear":
        return mlk.gemm_layoutA_linear(state["w"], state["x"], scale_matrix=state["scale"], bias=state["bias"])
    if kind == "chain":
        h = mlk.gemm_layoutABC(state["w1"], mlk.layoutB(state["x"]))
        return h, mlk.gemm_layoutAB_ContinuousC(state["w2"], h)
    return fused_moe(state["x"], state["w1"], state["w2"], state["logits"], state["case"]["picks"], **state["options"])


def work(case):
    """Weights, scales and activations read once, outputs written once; two operations per weight and token.  Of an
    expert layer, the experts that even routing of the tokens would be expected to reach."""
    tokens, size = case["tokens"], _BYTES[case["weights"]]

    def matrix(rows, k):
        return rows * k * size + (4 * math.ceil(rows / 128) * math.ceil(k / 128) if size == 1 else 0)

    if case["kind"] == "moe":
        e, picks, hidden, inter = case["experts"], case["picks"], case["hidden"], case["inter"]
        reached = e * (1 - (1 - picks / e) ** tokens)
        weights = reached * (matrix(2 * inter, hidden) + matrix(hidden, inter))
        return {"bytes": weights + 4 * tokens * hidden + 2 * tokens * e, "flops": 6 * tokens * picks * hidden * inter}
    rows, k = case["rows"], case["k"]
    if case["kind"] == "chain":
        rows2 = case["rows2"]
        return {"bytes": matrix(rows, k) + matrix(rows2, rows) + 2 * tokens * (k + rows + rows2),
                "flops": 2 * tokens * rows * (k + rows2)}
    return {"bytes": matrix(rows, k) + 2 * tokens * (k + rows), "flops": 2 * tokens * rows * k}


def tolerance(case):
    """Against the same path in 64 bits the results of one product are off by rel 1.66e-3, max 3.9e-3 in bf16 and by 2.1e-4,
    4.9e-4 in fp16 (the rounding of the output); the chain and the expert layers, which round once more in between, by
    2.4e-3, 1.1e-2 and 2.9e-4, 1.1e-3.  Four times that is allowed."""
    fp16 = case["weights"] == "fp16"
    if case["kind"] in ("chain", "moe"):
        return {"rel": 1.2e-3 if fp16 else 1e-2, "max": 4.5e-3 if fp16 else 0.043}
    return {"rel": 8.5e-4 if fp16 else 6.7e-3, "max": 2e-3 if fp16 else 0.016}
