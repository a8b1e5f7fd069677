"""The workloads this framework's speed is judged by.

Every case goes through the package's public entry points as a program that
serves or prepares a W4A16 model does:

* ``linear``      one or more layers' projections, ``w4a16_linear(x, packed,
                  scales)``: decode at one batch row, batched decode, prefill;
* ``mlp``         whole SwiGLU MLP blocks, ``mlp_decode``, the same range;
* ``quantize``    ``quantize_and_pack`` of an fp32 weight on the GPU (loading a
                  checkpoint);
* ``dequantize``  the way back, to fp32 or fp16 (export, evaluation).

A decode pass reads every weight once, and a model's weights never fit a
cache, so the small shapes run through several layers, each with its own
weights and its own hidden state, one call after another as a decode step
makes them: a pass then streams weights that have left the caches.

Sizes are the Llama projections that the benchmark and the tests use
(4096 x 4096, 11008 x 4096, 28672 x 8192 and 8192 x 28672, the 3584 x 8192
tensor-parallel shard), and ragged ones from the tests.
"""

import math
import sys
from pathlib import Path

import torch

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "decode-kernel_amd"))

from decode_kernel import dequantize, mlp_decode, quantize_and_pack, w4a16_linear  # noqa: E402

GROUP = 128
MAX_WEIGHTS = 28672 * 8192
MAX_FLOPS = 2.0 * 2048 * MAX_WEIGHTS
LAYER_BYTES = 128e6  # weights a multi-layer pass streams, about
MAX_LAYERS = 16


def listed():
    return [
        # Decode of one sequence: an attention projection of each of 16
        # layers. The smallest calls; launches and latency count.
        dict(name="linear_b1_4096x4096", op="linear", M=4096, K=4096, B=1, layers=16),
        # Decode of one sequence at the largest projection (70B gate or up).
        dict(name="linear_b1_28672x8192", op="linear", M=28672, K=8192, B=1, layers=1),
        # Batched decode at the longest rows (70B down).
        dict(name="linear_b16_8192x28672", op="linear", M=8192, K=28672, B=16, layers=1),
        # Batched decode, ragged: rows that fill no tile, an odd number of
        # groups per row, a batch over one tile.
        dict(name="linear_b20_5000x4224", op="linear", M=5000, K=4224, B=20, layers=12),
        # A busy server's decode batch, or the prefill of a short prompt.
        dict(name="linear_b128_11008x4096", op="linear", M=11008, K=4096, B=128, layers=6),
        # Prefill of a prompt whose length is no multiple of anything.
        dict(name="linear_b1000_4096x4096", op="linear", M=4096, K=4096, B=1000, layers=4),
        # Prefill of a long prompt at the largest projection.
        dict(name="linear_b2048_28672x8192", op="linear", M=28672, K=8192, B=2048, layers=1),
        # The MLP block in decode of one sequence (7B), in batched decode on
        # a tensor-parallel shard (70B over eight), and in prefill (7B).
        dict(name="mlp_b1_11008x4096", op="mlp", M=11008, K=4096, B=1, layers=3),
        dict(name="mlp_b8_3584x8192", op="mlp", M=3584, K=8192, B=8, layers=3),
        dict(name="mlp_b512_11008x4096", op="mlp", M=11008, K=4096, B=512, layers=1),
        # Loading: quantize one of a model's weights on the GPU.
        dict(name="quantize_11008x4096", op="quantize", M=11008, K=4096),
        # Export or evaluation: the weight back in floating point.
        dict(name="dequantize_4096x11008", op="dequantize", M=4096, K=11008, dtype="float32"),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _layers(weights):
    return max(1, min(MAX_LAYERS, int(LAYER_BYTES / (0.516 * weights))))


def draw(rng):
    """One more case: rows of 512-28672 (any number), 8 to 224 groups per row
    (odd counts among them), 1-2048 batch rows."""
    op = rng.choice(["linear"] * 5 + ["mlp"] * 3 + ["quantize", "dequantize"])
    while True:
        M = _log_int(rng, 512, 28672)
        K = GROUP * _log_int(rng, 8, 224)
        if op == "mlp":
            M = max(GROUP, M // GROUP * GROUP)  # the down projection's K
            if 3 * M * K > MAX_WEIGHTS:
                continue
        if M * K <= MAX_WEIGHTS:
            break
    if op == "quantize":
        return dict(op=op, M=M, K=K)
    if op == "dequantize":
        return dict(op=op, M=M, K=K, dtype=rng.choice(["float32", "float16"]))
    weights = (3 if op == "mlp" else 1) * M * K
    B = _log_int(rng, 1, 2048)
    layers = _layers(weights)
    while layers > 1 and 2.0 * B * weights * layers > MAX_FLOPS / 4:
        layers -= 1
    return dict(op=op, M=M, K=K, B=B, layers=layers)


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _weight(g, M, K):
    """A quantized weight (packed int32 [M, K/8], scales fp16 [M, K/128]) with
    the values that quantizing a Gaussian weight of std 0.02 gives: q about
    normal with std 2.6 in -7..7, scales around 0.02 * 2.7 / 7."""
    q = torch.randn(M, K // 8, 8, device="cuda", generator=g, dtype=torch.float16)
    q = (q * 2.6).round_().clamp_(-7, 7).to(torch.int8)
    packed = torch.zeros(M, K // 8, dtype=torch.int32, device="cuda")
    for n in range(8):
        packed |= (q[:, :, n].to(torch.int32) & 0xF) << (4 * n)
    spread = torch.randn(M, K // GROUP, device="cuda", generator=g)
    scales = (0.02 * 2.7 / 7 * (1 + 0.12 * spread).clamp_(0.5, 2.0)).half()
    return packed, scales


def _hidden(g, B, K):
    """A normalised hidden state."""
    return torch.randn(B, K, device="cuda", generator=g).half()


def prepare(case, seed):
    op, M, K = case["op"], case["M"], case["K"]
    g = _generator(seed)
    if op == "quantize":
        return dict(op=op, w=torch.randn(M, K, device="cuda", generator=g) * 0.02)
    if op == "dequantize":
        return dict(op=op, dtype=getattr(torch, case["dtype"]), layer=_weight(g, M, K))
    shapes = [(M, K)] if op == "linear" else [(M, K), (M, K), (K, M)]
    layers = [sum((_weight(g, m, k) for m, k in shapes), ()) for _ in range(case["layers"])]
    return dict(op=op, layers=layers, x=[_hidden(g, case["B"], K) for _ in layers])


def run(state):
    op = state["op"]
    if op == "linear":
        return [w4a16_linear(x, *layer) for x, layer in zip(state["x"], state["layers"])]
    if op == "mlp":
        return [mlp_decode(x, *layer) for x, layer in zip(state["x"], state["layers"])]
    if op == "quantize":
        return quantize_and_pack(state["w"])
    return dequantize(*state["layer"], dtype=state["dtype"])


def work(case):
    op, M, K = case["op"], case["M"], case["K"]
    weight = M * K / 2 + M * K / GROUP * 2
    if op == "quantize":
        return dict(bytes=4.0 * M * K + weight, flops=0)
    if op == "dequantize":
        return dict(bytes=weight + (4.0 if case["dtype"] == "float32" else 2.0) * M * K, flops=0)
    B, layers = case["B"], case["layers"]
    if op == "linear":
        return dict(bytes=layers * (weight + 2.0 * B * (M + K)), flops=layers * 2.0 * B * M * K)
    return dict(bytes=layers * (3 * weight + 2.0 * B * (K + K)), flops=layers * 6.0 * B * M * K)


def tolerance(case):
    """Quantizing and dequantizing are defined to the bit. The products sum in
    fp32 and round to fp16 once (twice in the MLP, whose hidden vector is
    fp16): 2.1e-4 (linear) and 2.9e-4 (MLP) from 64 bits in the 2-norm, which
    is that rounding, and at most half an fp16 step, 2^-11, at one value."""
    if case["op"] in ("quantize", "dequantize"):
        return "exact"
    return {"rel": 1e-3, "max": 6e-3}


def _dequantized(packed, scales):
    """The weight in 64 bits."""
    M, words = packed.shape
    w = torch.empty(M, words, 8, dtype=torch.float64, device=packed.device)
    for n in range(8):
        w[:, :, n] = ((packed << (28 - 4 * n)) >> 28).double()
    w = w.view(M, -1, GROUP)
    w *= scales.double()[:, :, None]
    return w.view(M, -1)


def exact(case, seed):
    state = prepare(case, seed)
    op = case["op"]
    if op == "quantize":
        w = state["w"].double().view(case["M"], -1, GROUP)
        return None, (w.abs().amax(-1) / 7).clamp_min(1e-8)
    if op == "dequantize":
        return _dequantized(*state["layer"])
    out = []
    for x, layer in zip(state["x"], state["layers"]):
        x = x.double()
        if op == "linear":
            out.append(x @ _dequantized(*layer).T)
            continue
        gate = x @ _dequantized(*layer[0:2]).T
        up = x @ _dequantized(*layer[2:4]).T
        out.append((torch.nn.functional.silu(gate) * up) @ _dequantized(*layer[4:6]).T)
    return out
