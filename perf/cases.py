"""The work that programs built on this framework have it do, as timed cases.

A case is one layer or one small net, called through the public entry points
the way a user's program calls them:

* ``mlir_edsl_hip.device.dense_launch`` on tensors that live in HBM (the
  caller owns the output buffers and the stream), in f32 and in i32;
* ``MLIRCompiler.execute_gpu_function`` on host arrays, with the net's weights
  bound as device-resident parameters, for a serving program behind the
  reference's front end.

The framework is an inference path (no gradients), so a pass is a forward
pass. Sizes come from this repository's workloads, tests and benchmark, or are
generic; ``draw`` spreads over the same ranges, odd sizes included.
"""
from __future__ import annotations

import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.getcwd(), "ml-edsl_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from mlir_edsl_hip import _native, wire  # noqa: E402
from mlir_edsl_hip._mlir_backend import MLIRCompiler  # noqa: E402
from mlir_edsl_hip.device import dense_launch  # noqa: E402

# Epilogue names: what the layer does after X @ W.
EPILOGUES = {
    "none": _native.EPI_NONE,
    "relu": _native.EPI_RELU,
    "bias": _native.EPI_BIAS,
    "bias_relu": _native.EPI_BIAS_RELU,
    "bias_leaky": _native.EPI_BIAS_LEAKY,
    "bias_if_relu": _native.EPI_BIAS_IF_RELU,
}
ALPHA = 0.01  # slope of the leaky epilogue

# Largest work of a drawn case: the largest listed layer, and the bytes of the
# largest listed weight matrix with its activations.
MAX_FLOPS = 2 * 4096 ** 3
MAX_BYTES = 4 * (8192 * 8192 + 4 * 16 * 8192)


def listed():
    return [
        # The smallest calls: a three-layer classifier head on a small batch,
        # one launch after the other, where latency and launches are the time.
        {"name": "mlp_small", "kind": "mlp", "M": 64, "widths": "256,256,256,64"},
        # A plain linalg.matmul at a middle size of the reference's benchmarks.
        {"name": "matmul_512", "kind": "dense", "M": 512, "K": 512, "N": 512, "epi": "none"},
        # The reference's largest GPU benchmark layer.
        {"name": "dense_1024", "kind": "dense", "M": 1024, "K": 1024, "N": 1024, "epi": "bias_relu"},
        # A layer no tile divides, with the leaky activation.
        {"name": "dense_1000_leaky", "kind": "dense", "M": 1000, "K": 1000, "N": 1000, "epi": "bias_leaky"},
        # The largest layer: the headline workload.
        {"name": "dense_4096", "kind": "dense", "M": 4096, "K": 4096, "N": 4096, "epi": "bias_relu"},
        # Odd in every size, so no row is 16-byte aligned.
        {"name": "matmul_relu_2001", "kind": "dense", "M": 2001, "K": 2001, "N": 2001, "epi": "relu"},
        # A long batch through a narrow layer: many rows, short K.
        {"name": "dense_tall", "kind": "dense", "M": 10000, "K": 500, "N": 1000, "epi": "bias_if_relu"},
        # A decode-sized batch against a large weight matrix: HBM-bound.
        {"name": "small_batch_8192", "kind": "dense", "M": 16, "K": 8192, "N": 8192, "epi": "bias_relu"},
        # A few rows more and an odd output width.
        {"name": "small_batch_odd", "kind": "dense", "M": 48, "K": 4096, "N": 4097, "epi": "bias"},
        # An integer layer on quantised (int8-valued) i32 tensors.
        {"name": "int_2048", "kind": "int", "M": 2048, "K": 2048, "N": 2048},
        # Two integer layers: the second reads the first one's i32 activations,
        # which are wider than int8.
        {"name": "int_net", "kind": "int_net", "M": 512, "widths": "1024,1024,512"},
        # Serving behind the reference's front end: host arrays in and out,
        # weights resident on the device.
        {"name": "host_net", "kind": "host_net", "M": 256, "widths": "1024,1024,1024,256"},
    ]


def _log_int(rng, lo, hi):
    """An integer from [lo, hi], spread over its logarithm; mostly odd or ragged
    values, and every third one rounded to a multiple of 64 as layer widths often are."""
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    if rng.randrange(3) == 0:
        v = max(lo, min(hi, (v + 32) // 64 * 64))
    return max(lo, min(hi, v))


def draw(rng):
    kind = rng.choice(["mlp", "dense", "dense", "dense", "small", "small", "int", "int_net", "host_net"])
    while True:
        if kind == "dense":
            c = {"kind": "dense", "M": _log_int(rng, 65, 10000), "K": _log_int(rng, 64, 4096),
                 "N": _log_int(rng, 64, 4096), "epi": rng.choice(sorted(EPILOGUES))}
        elif kind == "small":
            c = {"kind": "dense", "M": _log_int(rng, 1, 64), "K": _log_int(rng, 512, 8192),
                 "N": _log_int(rng, 512, 8192), "epi": rng.choice(sorted(EPILOGUES))}
        elif kind == "int":
            c = {"kind": "int", "M": _log_int(rng, 64, 4096), "K": _log_int(rng, 64, 4096),
                 "N": _log_int(rng, 64, 4096)}
        else:
            n = rng.randrange(2, 4) if kind == "int_net" else rng.randrange(2, 5)
            hi = 512 if kind == "mlp" else 2048
            c = {"kind": kind, "M": _log_int(rng, 1, 1024 if kind == "int_net" else 512),
                 "widths": ",".join(str(_log_int(rng, 32, hi)) for _ in range(n))}
        w = work(c)
        if w["flops"] <= MAX_FLOPS and w["bytes"] <= MAX_BYTES:
            return c


def _widths(case):
    """The widths of a net: its input's, then each layer's output's."""
    if "widths" in case:
        return [int(v) for v in case["widths"].split(",")]
    return [case["K"], case["N"]]


def _is_int(case):
    return case["kind"] in ("int", "int_net")


def _epis(case):
    """The epilogue of each layer: hidden layers bias + ReLU, a net's last layer bias only."""
    n = len(_widths(case)) - 1
    if case["kind"] == "dense":
        return [case["epi"]]
    if _is_int(case):
        return ["bias_relu"] * n
    return ["bias_relu"] * (n - 1) + ["bias"]


def _host_layer(rng, K, N):
    W = (rng.standard_normal((K, N), dtype=np.float32) / np.float32(math.sqrt(K))).astype(np.float32)
    b = (rng.random(N, dtype=np.float32) * np.float32(0.2) - np.float32(0.1)).astype(np.float32)
    return W, b


def _inputs(case, seed):
    """X and the layers' (W, b): N(0, 1) activations, N(0, 1/K) weights and U[-0.1, 0.1)
    biases; for integers 4-bit values and 10-bit biases, as the repository's workloads draw them."""
    w = _widths(case)
    M = case["M"]
    if case["kind"] == "host_net":
        rng = np.random.default_rng(seed)
        X = rng.standard_normal((M, w[0]), dtype=np.float32)
        return X, [_host_layer(rng, k, n) for k, n in zip(w, w[1:])]
    g = torch.Generator(device="cuda").manual_seed(seed)
    layers = []
    if _is_int(case):
        def ints(shape, lo, hi):
            return torch.randint(lo, hi, shape, device="cuda", dtype=torch.int32, generator=g)
        X = ints((M, w[0]), -8, 8)
        for k, n in zip(w, w[1:]):
            layers.append((ints((k, n), -8, 8), ints((n,), -512, 512)))
    else:
        X = torch.randn(M, w[0], device="cuda", generator=g)
        for k, n in zip(w, w[1:]):
            W = torch.randn(k, n, device="cuda", generator=g).div_(math.sqrt(k))
            layers.append((W, torch.rand(n, device="cuda", generator=g).mul_(0.2).sub_(0.1)))
    return X, layers


def prepare(case, seed):
    """Inputs, weights and what a program keeps between calls: its output and
    activation buffers, or the compiled function with its weights bound."""
    X, layers = _inputs(case, seed)
    epis = _epis(case)
    if case["kind"] == "host_net":
        w = _widths(case)
        comp = MLIRCompiler()
        comp.set_target("gpu")
        prog = [wire.Layer(f"W{i}", n, f"b{i}", "relu" if e == "bias_relu" else "none")
                for i, (n, e) in enumerate(zip(w[1:], epis))]
        comp.compile_function(wire.dense_program("net", ("X", case["M"], w[0]), prog))
        arrays = [X]
        for i, (W, b) in enumerate(layers):
            comp.bind_parameter("net", f"W{i}", W)
            comp.bind_parameter("net", f"b{i}", b)
            arrays += [W, b]
        return {"host": True, "comp": comp, "arrays": arrays, "out": [case["M"], w[-1]]}
    steps = []
    x = X
    for (W, b), e in zip(layers, epis):
        y = torch.empty(x.shape[0], W.shape[1], dtype=x.dtype, device="cuda")
        code = EPILOGUES[e]
        steps.append((x, W, b if code & 1 else None, y, code))
        x = y
    return {"host": False, "steps": steps}


def run(state):
    if state["host"]:
        args = [(a.ctypes.data, list(a.shape)) for a in state["arrays"]]
        raw = state["comp"].execute_gpu_function("net", args, state["out"], 4)
        return np.frombuffer(raw, np.float32).reshape(state["out"])
    for x, W, b, y, code in state["steps"]:
        dense_launch(x, W, b, y, code, ALPHA)
    return y


def work(case):
    """Each layer's weights and bias, the net's input and its output once; 2 M N K operations
    a layer. Activations between layers are counted out: a path could keep them on the chip."""
    w = _widths(case)
    M = case["M"]
    nbytes, flops = M * w[0] + M * w[-1], 0
    for k, n, e in zip(w, w[1:], _epis(case)):
        nbytes += k * n + (n if EPILOGUES[e] & 1 else 0)
        flops += 2 * M * n * k
    return {"bytes": 4 * nbytes, "flops": flops}


def tolerance(case):
    """Integers are exact. f32: rounding of a K-term sum grows with sqrt(K); see the constants."""
    if _is_int(case):
        return "exact"
    K = max(_widths(case)[:-1])
    depth = len(_widths(case)) - 1
    rel = REL_1024 * math.sqrt(max(K, 64) / 1024) * math.sqrt(depth)
    return {"rel": rel, "max": 16 * rel}


# Measured against float64 at K = 1024: relative 2-norm error 2.9e-7 here and 5.7e-7 for torch's fp32
# product (another order of summation), largest difference up to 15 times that; times about four.
REL_1024 = 2e-6


def exact(case, seed):
    X, layers = _inputs(case, seed)
    if case["kind"] == "host_net":
        X = torch.from_numpy(X)
        layers = [(torch.from_numpy(W), torch.from_numpy(b)) for W, b in layers]
        if torch.cuda.is_available():
            X, layers = X.cuda(), [(W.cuda(), b.cuda()) for W, b in layers]
    h = X.double()
    for (W, b), e in zip(layers, _epis(case)):
        h = h @ W.double()  # integers: sums stay far below 2^53, so this is exact
        code = EPILOGUES[e]
        if code & 1:
            h = h + b.double()
        if _is_int(case):  # i32 tensors: wrap modulo 2^32
            h = torch.remainder(h + 2.0 ** 31, 2.0 ** 32) - 2.0 ** 31
        act = code >> 1
        if act in (1, 3):
            h = h.clamp_min(0.0)
        elif act == 2:
            h = torch.where(h > 0, h, h * float(np.float32(ALPHA)))
    if case["kind"] == "host_net":
        return h.cpu().numpy()
    return h.to(torch.int32) if _is_int(case) else h
