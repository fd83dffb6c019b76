"""What the operators of this package are measured on: one pass of each listed case through the public modules and
callables, as a training or an inference program calls them.

A case names an operator, a dense (batch, rows, cols) input, its storage type and whether the pass trains (forward
and backward; the input's and the parameters' gradients come back) or infers (forward alone, under no_grad).
"""
import math
import os
import random
import sys

import torch

_PACKAGE = os.path.join(os.getcwd(), "triton-hub_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

from TritonHub import Activations, Layers, Normalization, Ops  # noqa: E402
from TritonHub.Normalization import fused  # noqa: E402

DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
BYTES = {"bf16": 2, "f16": 2, "f32": 4}
ACTIVATIONS = {"gelu": lambda: Activations.GeLU(), "gelu_tanh": lambda: Activations.GeLU(approximate="tanh"),
               "silu": lambda: Activations.SiLU(), "relu": lambda: Activations.ReLU(), "sigmoid": lambda: Activations.Sigmoid(),
               "mish": lambda: Activations.Mish()}
NORMS = ("layernorm", "rmsnorm", "layernorm+gelu", "rmsnorm+silu")


def _case(name, op, batch, rows, cols, dtype, train=True, p=0.0):
    return {"name": name, "op": op, "batch": batch, "rows": rows, "cols": cols, "dtype": dtype, "train": train, "p": p}


def listed():
    return [
        # the README's first example: a float32 LayerNorm over a handful of tokens, where host work and launches are all there is
        _case("layernorm_f32_2x100x128", "layernorm", 2, 100, 128, "f32"),
        # one decoding step of a served language model: 64 sequences, one token each, no gradients
        _case("rmsnorm_decode_bf16_64x4096", "rmsnorm", 64, 1, 4096, "bf16", train=False),
        # a training step's norm over 16384 tokens of a 4096-wide model: the workload of bench.py
        _case("rmsnorm_bf16_16384x4096", "rmsnorm", 4, 4096, 4096, "bf16"),
        # the widest training batch of the contract configurations
        _case("layernorm_bf16_32768x8192", "layernorm", 8, 4096, 8192, "bf16"),
        # rows that are no power of two and start off cache lines, in float16
        _case("layernorm_f16_8192x6000", "layernorm", 2, 4096, 6000, "f16"),
        # query / key norms: one short row per token and head (16 x 1024 tokens, 32 heads of 128)
        _case("rmsnorm_heads_bf16_524288x128", "rmsnorm", 16, 32768, 128, "bf16"),
        # the norm in front of a feed-forward block with its activation in the same pass
        _case("layernorm_gelu_bf16_16384x4096", "layernorm+gelu", 4, 4096, 4096, "bf16"),
        # attention rows of a vision transformer: 197 tokens, 64 images, 12 heads
        _case("softmax_bf16_768x197x197", "softmax", 768, 197, 197, "bf16"),
        # token log-probabilities over a 128256-word vocabulary
        _case("logsoftmax_bf16_4096x128256", "logsoftmax", 1, 4096, 128256, "bf16"),
        # a batch of embeddings brought to unit length before a contrastive loss
        _case("normalize_f16_65536x1024", "normalize", 64, 1024, 1024, "f16", p=2.0),
        # the activation of a feed-forward block
        _case("gelu_bf16_16384x4096", "gelu", 4, 4096, 4096, "bf16"),
        # dropout on a residual stream
        _case("dropout_bf16_16384x4096", "dropout", 4, 4096, 4096, "bf16", p=0.1),
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _width(rng, low, high, step=128):
    """A model width: mostly a multiple of `step`, now and then any number."""
    n = _log(rng, low, high)
    return max(step, n // step * step) if rng.random() < 0.7 else n


def draw(rng):
    kind = rng.choice(("block", "block", "decode", "heads", "fused", "attention", "vocabulary", "embedding", "activation", "dropout"))
    dtype = rng.choice(("bf16", "bf16", "bf16", "f16", "f32"))
    train, p, batch = True, 0.0, 1
    most = 2 ** 26 if dtype == "f32" else 2 ** 27            # elements of the input

    if kind == "block":                                      # norms of a transformer block, from a short prompt to a full batch
        op, cols, rows = rng.choice(("layernorm", "rmsnorm")), _width(rng, 256, 16384), _log(rng, 128, 32768)
    elif kind == "decode":                                   # inference: one token per sequence, or a short prefill
        op, cols, rows, train = rng.choice(("layernorm", "rmsnorm")), _width(rng, 1024, 8192), _log(rng, 1, 512), False
    elif kind == "heads":                                    # norms over the columns of one attention head
        op, cols, rows = rng.choice(("layernorm", "rmsnorm")), rng.choice((32, 64, 80, 96, 128, 256)), _log(rng, 1024, 2 ** 20)
    elif kind == "fused":
        op, cols, rows = rng.choice(("layernorm+gelu", "rmsnorm+silu")), _width(rng, 256, 8192), _log(rng, 128, 16384)
    elif kind == "attention":                                # (batch * heads, queries, keys): square, any length
        op, cols, batch = "softmax", _log(rng, 32, 4096), _log(rng, 16, 1024)
        rows = cols
    elif kind == "vocabulary":
        op, cols, rows = rng.choice(("logsoftmax", "logsoftmax", "softmax")), _log(rng, 30000, 262144), _log(rng, 16, 4096)
    elif kind == "embedding":
        op, cols, rows = "normalize", _width(rng, 3, 4096, 16), _log(rng, 512, 2 ** 20)
        p = rng.choice((2.0, 2.0, 2.0, 1.0, 3.0))
    elif kind == "activation":
        op, cols, rows = rng.choice(tuple(ACTIVATIONS)), _width(rng, 256, 16384), _log(rng, 128, 32768)
    else:
        op, cols, rows, p = "dropout", _width(rng, 256, 16384), _log(rng, 128, 32768), rng.choice((0.1, 0.2, 0.5))
    batch = max(1, min(batch, most // (rows * cols)))
    rows = max(1, min(rows, most // (batch * cols)))
    case = _case("", op, batch, rows, cols, dtype, train, p)
    del case["name"]
    return case


def prepare(case, seed):
    device = torch.device("cuda", 0)
    dtype, shape, n, op = DTYPES[case["dtype"]], (case["batch"], case["rows"], case["cols"]), case["cols"], case["op"]
    gen = torch.Generator(device=device).manual_seed(seed)

    def normal(*size, scale=1.0, offset=0.0):
        return torch.randn(*size, device=device, dtype=dtype, generator=gen).mul_(scale).add_(offset)

    # activations with a spread and an offset of their own; logits and attention scores a few units wide
    x = normal(*shape, scale=3.0) if op in ("softmax", "logsoftmax") else normal(*shape, scale=1.5, offset=0.25)
    dy = normal(*shape) if case["train"] else None
    if op in NORMS:
        if op == "layernorm":
            module = Normalization.LayerNorm(n, device=device, dtype=dtype)
        elif op == "rmsnorm":
            module = Normalization.RMSNorm(n, device=device, dtype=dtype)
        elif op == "layernorm+gelu":
            module = fused.LayerNormActivation(n, activation="gelu", device=device, dtype=dtype)
        else:
            module = fused.RMSNormActivation(n, activation="silu", device=device, dtype=dtype)
        with torch.no_grad():
            module.weight.copy_(normal(n, scale=0.1, offset=1.0))
            if module.bias is not None:
                module.bias.copy_(normal(n, scale=0.1))
        parameters = list(module.parameters())
    else:
        parameters = []
        if op == "dropout":
            module = Layers.Dropout(case["p"])
        elif op == "normalize":
            module = Ops.normalize(p=case["p"])
        elif op == "softmax":
            module = Activations.Softmax()
        elif op == "logsoftmax":
            module = Activations.LogSoftmax()
        else:
            module = ACTIVATIONS[op]()
    x.requires_grad_(case["train"])
    return {"module": module, "x": x, "dy": dy, "wanted": [x] + parameters, "mask_seed": seed if op == "dropout" else None}


def run(state):
    if state["mask_seed"] is not None:
        random.seed(state["mask_seed"])          # the mask of a dropout follows from Python's random numbers
    if state["dy"] is None:
        with torch.no_grad():
            return state["module"](state["x"])
    y = state["module"](state["x"])
    return (y,) + torch.autograd.grad(y, state["wanted"], state["dy"])


# Operations per element of a forward + backward (and of a forward alone): reductions, the affine part, exponentials as one.
_OPERATIONS = {"layernorm": (22, 8), "rmsnorm": (15, 5), "layernorm+gelu": (60, 24), "rmsnorm+silu": (35, 12), "softmax": (8, 5),
               "logsoftmax": (8, 5), "normalize": (8, 3), "gelu": (36, 16), "gelu_tanh": (24, 10), "silu": (10, 4), "relu": (2, 1),
               "sigmoid": (6, 3), "mish": (20, 8), "dropout": (110, 55)}       # dropout: ten Philox rounds per element and pass


def work(case):
    m, n, s, op = case["batch"] * case["rows"], case["cols"], BYTES[case["dtype"]], case["op"]
    # forward: x in, y out.  Backward: one more tensor and dy in, dx out; a dropout reads nothing but dy.  normalize by
    # another p than 1 and 2 needs x and y.
    passes = 2 if not case["train"] else 4 if op == "dropout" else 6 if op == "normalize" and case["p"] not in (1.0, 2.0) else 5
    total = passes * m * n * s
    if op in NORMS:
        statistics = 2 if op.startswith("layernorm") else 1          # float32 per row; gamma alone or gamma and beta
        total += (2 if case["train"] else 1) * statistics * (4 * m + n * s) + (n * s if case["train"] else 0)
    if op == "normalize":
        total += 2 * m * s
    return {"bytes": total, "flops": _OPERATIONS[op][0 if case["train"] else 1] * m * n}


def tolerance(case):
    """About four times the distance between a pass and the same operator in float64 (largest over the outputs, on rows
    of 300, 1000 and 128256 columns): relative error 1.7e-3 in bfloat16 (3.1e-3 where a gradient is a difference of
    rounded outputs), 2.1e-4 (3.9e-4) in float16, 1.5e-7 in float32; largest single difference 3.9e-3, 4.9e-4, 4e-7,
    of those gradients 7.9e-2, 1.2e-2 and 9e-6."""
    if case["op"] == "dropout":
        return "exact"                           # the mask and the scaled values are defined bit for bit
    from_outputs = case["op"] in ("softmax", "logsoftmax", "normalize", "sigmoid")
    return {"bf16": {"rel": 1e-2, "max": 0.3 if from_outputs else 0.03},
            "f16": {"rel": 1.5e-3, "max": 0.05 if from_outputs else 4e-3},
            "f32": {"rel": 1e-6, "max": 4e-5 if from_outputs else 4e-6}}[case["dtype"]]
