"""The work this framework is measured on: single linear layers and products through its public entry
points (``FastLinear``, ``mm_t``, ``matmul``, ``patch``), from one decoded token to a BERT-base batch.

Three entry points are timed, as ``entry`` in a case:

* ``mm_t``: the functional product ``mm_t(x, w_t, bias, out_dtype)`` on a [K, N] fp16 weight;
* ``linear``: a ``FastLinear`` layer made from an ``nn.Linear``, called on its activations;
* ``matmul``: ``gtx16_fp16.matmul`` of two fp16 matrices;
* ``mlp``: a transformer feed-forward block (Linear, GELU, Linear) whose layers ``patch`` replaced.

``x`` and ``out`` name the activation and output types, ``M`` the rows (tokens), ``K`` and ``N`` the
layer's in and out features. ``outliers`` scales 1 % of the rows (at least one) up to a largest
magnitude in [2e3, 2e5] (fp16: [2e3, 8e3], so that fp16 outputs stay finite), the massive
activations the per-row rescale exists for. ``decode_copy`` turns on the layer's opt-in decode layout.
"""
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "gtx16-fp16_amd"))

import gtx16_fp16 as g  # noqa: E402

DTYPES = {"f32": torch.float32, "f16": torch.float16}
SIZE = {"f32": 4, "f16": 2}

# No listed or drawn case asks for more than the feed-forward block of a BERT-base batch does.
MAX_FLOPS = 4 * 65536 * 768 * 3072 // 2   # one of its two layers
MAX_ACTIVATIONS = 65536 * (768 + 3072)     # elements of such a layer's input and output


def _case(entry, M, K, N, x="f32", out="f32", bias=True, outliers=False, decode_copy=False, name=None):
    c = {"entry": entry, "M": M, "K": K, "N": N, "x": x, "out": out, "bias": bias, "outliers": outliers,
         "decode_copy": decode_copy}
    if name is not None:
        c["name"] = name
    return c


def listed():
    return [
        # token-by-token generation in a small fp32 model: one token through a 1024-wide projection,
        # where the launch and the host path count for more than the 2 MiB weight
        _case("linear", 1, 1024, 1024, name="decode_layer_1024"),
        # one token against a 4096 x 4096 weight, the memory-bound product decoding consists of
        _case("mm_t", 1, 4096, 4096, bias=False, name="decode_product_4096"),
        # four sequences decoded together in a half-precision model
        _case("linear", 4, 4096, 4096, x="f16", out="f16", name="decode_batch4_fp16"),
        # seven sequences into a 4096 -> 11008 feed-forward projection, fp32 activations
        _case("mm_t", 7, 4096, 11008, name="decode_batch7_wide"),
        # a serving batch of 64 single tokens (or a short prompt), long reduction, few columns
        _case("linear", 64, 4096, 1024, name="batch64_4096_1024"),
        # the fp16 matrix product of a script or an attention block: torch.matmul's drop-in
        _case("matmul", 1024, 1024, 1024, x="f16", out="f16", bias=False, name="matmul_1024"),
        # a prompt of 333 tokens in an fp32 model, one of them with massive activations
        _case("linear", 333, 4096, 4096, outliers=True, name="prompt333_outliers"),
        # a prompt of 777 tokens into a wide feed-forward projection, half precision
        _case("linear", 777, 3072, 8192, x="f16", out="f16", name="prompt777_fp16"),
        # the square product with 1 % outlier rows, fp32 in and out: the benchmark's workload
        _case("mm_t", 4096, 4096, 4096, outliers=True, name="square_4096_outliers"),
        # a long half-precision batch against a 2048 x 2048 weight (the reference's GEMM sweep)
        _case("matmul", 8192, 2048, 2048, x="f16", out="f16", bias=False, name="matmul_8192_2048"),
        # BERT-base, 256 x 256 tokens: the attention output projection (Q, K and V have its shape)
        _case("linear", 65536, 768, 768, name="bert_projection"),
        # ... and its feed-forward block as `patch` leaves it
        _case("mlp", 65536, 768, 3072, name="bert_feed_forward"),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def _features(rng, hi=14336):
    # layer widths: multiples of 8, half of them multiples of 128 (as most models' are)
    n = _log_uniform(rng, 256, hi)
    step = 128 if rng.random() < 0.5 else 8
    return max(256, n // step * step)


def draw(rng):
    kind = rng.choice(["decode", "batch", "prompt", "large"])
    rows = {"decode": (1, 8), "batch": (9, 96), "prompt": (65, 1500), "large": (1024, 65536)}[kind]
    while True:
        M = _log_uniform(rng, *rows)
        K, N = _features(rng), _features(rng)
        if 2 * M * K * N <= MAX_FLOPS and M * (K + N) <= MAX_ACTIVATIONS and K * N <= 4096 * 14336:
            break
    entry = rng.choice(["mm_t", "linear", "linear", "matmul"])
    x = "f16" if entry == "matmul" else rng.choice(["f32", "f32", "f16"])
    out = x if entry != "mm_t" else rng.choice(["f32", "f16"])
    outliers = rng.random() < 0.25
    if out == "f16" and x == "f32":
        outliers = False  # their outputs would leave fp16's range
    return _case(entry, M, K, N, x=x, out=out, bias=entry != "matmul" and rng.random() < 0.7, outliers=outliers,
                 decode_copy=entry == "linear" and kind == "decode" and rng.random() < 0.25)


def _randn(gen, *shape, scale=1.0):
    return torch.randn(*shape, generator=gen, device="cuda") * scale


def _inputs(case, seed):
    """x in the case's type, then per layer (w [K, N] fp32 holding fp16 values, bias fp32 or None)."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    M, K, N = case["M"], case["K"], case["N"]
    x = _randn(gen, M, K)
    if case["outliers"]:
        n = max(1, round(0.01 * M))
        rows = torch.randperm(M, generator=gen, device="cuda")[:n]
        hi = 2e5 if case["x"] == "f32" else 8e3
        top = 2e3 + (hi - 2e3) * torch.rand(n, 1, generator=gen, device="cuda")
        x[rows] *= top / x[rows].abs().amax(1, keepdim=True)
    layers = []
    for k, n in [(K, N), (N, K)] if case["entry"] == "mlp" else [(K, N)]:
        w = _randn(gen, k, n, scale=0.02).half().float()
        b = _randn(gen, n, scale=0.02) if case["bias"] else None
        layers.append((w, b))
    return x.to(DTYPES[case["x"]]), layers


def _nn_linear(w, b):
    lin = torch.nn.Linear(w.shape[0], w.shape[1], bias=b is not None, device="meta")
    lin.weight = torch.nn.Parameter(w.t(), requires_grad=False)
    if b is not None:
        lin.bias = torch.nn.Parameter(b, requires_grad=False)
    return lin


def prepare(case, seed):
    x, layers = _inputs(case, seed)
    state = {"case": case, "x": x}
    if case["entry"] == "mlp":
        (w1, b1), (w2, b2) = layers
        state["model"] = torch.nn.Sequential(_nn_linear(w1, b1), torch.nn.GELU(), _nn_linear(w2, b2))
        g.patch(state["model"])
    elif case["entry"] == "linear":
        state["model"] = g.FastLinear.from_linear(_nn_linear(*layers[0]))
        state["model"].prepack_decode = case["decode_copy"]
    else:
        w, b = layers[0]
        state["w_t"], state["bias"] = w.half(), b
    return state


def run(state):
    case = state["case"]
    if case["entry"] in ("linear", "mlp"):
        return state["model"](state["x"])
    if case["entry"] == "matmul":
        return g.matmul(state["x"], state["w_t"])
    return g.mm_t(state["x"], state["w_t"], state["bias"], DTYPES[case["out"]])


def work(case):
    M, K, N = case["M"], case["K"], case["N"]
    if case["entry"] == "mlp":
        return {"bytes": 2 * M * K * 4 + 2 * 2 * K * N + 4 * (K + N), "flops": 4 * M * K * N}
    return {"bytes": M * K * SIZE[case["x"]] + 2 * K * N + (4 * N if case["bias"] else 0) + M * N * SIZE[case["out"]],
            "flops": 2 * M * K * N}


def tolerance(case):
    # About four times the error against 64 bits of the paths as measured: 2.1e-4 for one rounding of
    # the activations (M > 8, fp32 activations) or of the outputs to fp16, 3.0e-4 for the feed-forward
    # block, which rounds its input and its hidden activations; else fp32 sums (at most 1e-5).
    if case["entry"] == "mlp":
        return {"rel": 1.2e-3}
    if case["out"] == "f16" or (case["M"] > 8 and case["x"] == "f32"):
        return {"rel": 8.5e-4}
    return {"rel": 1e-5}


def exact(case, seed):
    x, layers = _inputs(case, seed)
    y = x.double()
    for i, (w, b) in enumerate(layers):
        if i:
            y = torch.nn.functional.gelu(y)
        y = y @ w.double()
        if b is not None:
            y += b.double()
    return y
