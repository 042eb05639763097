"""The calls a user of this framework makes, as cases that can be timed and whose outputs can be compared.

Each case is one pass through a public entry point, on inputs made on the GPU from a seed:

  linear     MixedLinear on [batch, seq, K] activations: the layer a model is built from, decode to prefill
  graph      the four projections of one decoder layer, MixedLinear each, captured once and replayed as a HIP graph
  module     the extension module `mixedgemm`: reorder_quantize_x, then matmul on row-major weights, each blocking
  quantize   reorder_quantize_x into buffers the caller keeps (activations handed to several GEMMs)
  pack       PackedWeights.from_float: a layer's bf16 weights quantized and put in the order the GEMM reads
  calibrate  calibrate_reorder_index: the channel order of a layer from a sample of its activations

Activations are N(0, 1) with K/32 outlier channels thirty times as large, weights N(0, 0.02), as in bench.py.
"""
import importlib
import math
import os
import sys

import torch

import mixedgemm_amd
from mixedgemm_amd import abi, linear

DEV = "cuda"
EPS = 1e-5

# `plan`: how K is split over the activation formats. "default": linear.default_split (MXFP4 + MXFP6 + MXFP8);
# "fp4": all MXFP4; "fp4_fp8": MXFP4 with 128 MXFP8 outlier channels.
LISTED = (
    # One sequence decoding: a square projection for a single token. Launches and host time count.
    dict(name="decode_1_token", op="linear", m=1, n=4096, k=4096, plan="default", norm=False, bias=False),
    # Eight sequences decoding: the wide up-projection behind its RMSNorm. Weight bytes against launches.
    dict(name="decode_8_up_norm", op="linear", m=8, n=14336, k=4096, plan="default", norm=True, bias=False),
    # A serving loop: one decoder layer's projections (qkv, output, gate + up, down) for 16 sequences, as a graph.
    dict(name="decode_16_layer_graph", op="graph", m=16, n=14336, k=4096, plan="default", norm=True, bias=False),
    # A batch of 32 through the long-K down-projection: few tokens, segments that end in half a matrix step.
    dict(name="batch_32_down", op="linear", m=32, n=4096, k=14336, plan="default", norm=False, bias=False),
    # A short prompt, or a large decode batch, through a square projection with a bias.
    dict(name="batch_128_bias", op="linear", m=128, n=4096, k=4096, plan="default", norm=False, bias=True),
    # The reference's own benchmark shape (bench_reorder_gemm.cu:24-29), through the reference's operator surface.
    dict(name="module_1024", op="module", m=1024, n=4096, k=4096, plan="default", norm=False, bias=False),
    # Ragged: a token count that is no multiple of anything, a feature count that is not whole tiles, a bias, and
    # the plan without MXFP6 and MXFP8.
    dict(name="ragged_777_fp4_bias", op="linear", m=777, n=5000, k=5120, plan="fp4", norm=False, bias=True),
    # Prefill, long K: the down-projection of 2048 tokens.
    dict(name="prefill_2048_down", op="linear", m=2048, n=4096, k=14336, plan="default", norm=False, bias=False),
    # Prefill, the largest: 4096 tokens through the RMSNorm and the wide up-projection.
    dict(name="prefill_4096_up_norm", op="linear", m=4096, n=14336, k=4096, plan="default", norm=True, bias=False),
    # Activations of a prefill quantized on their own.
    dict(name="quantize_4096", op="quantize", m=4096, n=0, k=4096, plan="default", norm=False, bias=False),
    # Loading a model: one wide layer's weights.
    dict(name="pack_14336", op="pack", m=0, n=14336, k=4096, plan="default", norm=False, bias=False),
    # Calibrating a layer on a sample of 4096 tokens.
    dict(name="calibrate_4096", op="calibrate", m=4096, n=0, k=4096, plan="default", norm=False, bias=False),
)

#: 2 M N K of the largest listed case: no drawn one costs more.
_MOST = 2 * 4096 * 14336 * 4096
_OPS = ("linear",) * 7 + ("graph", "module", "quantize", "pack", "calibrate")


def listed():
    return [dict(c) for c in LISTED]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_k(rng):
    """Input channels: one of the widths the reference instantiates its quantizers for, or any multiple of 32."""
    if rng.random() < 0.5:
        return rng.choice(linear.REFERENCE_K)
    return _log_int(rng, 1024 // 32, 18944 // 32) * 32


def _draw_n(rng, step, most=18944):
    """Output features: whole 128s mostly, multiples of 8, or (step 1) any count. Above 256, where packing pads."""
    shape = rng.random()
    if shape < 0.6:
        return _log_int(rng, 3, most // 128) * 128
    if shape < 0.85 or step > 1:
        return _log_int(rng, 34, most // 8) * 8
    return _log_int(rng, 257, most)


def draw(rng):
    op = rng.choice(_OPS)
    k = _draw_k(rng)
    m, n, plan, norm, bias = 0, 0, "default", False, False
    if op == "linear":
        n = _draw_n(rng, 1)
        m = _log_int(rng, 1, max(1, min(8192, _MOST // (2 * n * k))))
        norm, bias = rng.random() < 0.35, rng.random() < 0.35
        if k % 128 == 0 and rng.random() < 0.25:
            plan = rng.choice(("fp4", "fp4_fp8"))
    elif op == "graph":
        k = rng.choice((2048, 3584, 4096, 5120))
        n = k * rng.choice((2, 3, 4)) // 128 * 128
        m, norm = _log_int(rng, 1, 64), True
    elif op == "module":
        n = _draw_n(rng, 8)   # the reference's GEMMs store eight features at a time
        m = _log_int(rng, 1, max(1, min(8192, _MOST // (2 * n * k))))
    elif op == "pack":
        k = max(1024, k // 128 * 128)
        n = _draw_n(rng, 1, min(18944, 14336 * 4096 // k))
        if any(seg % 128 for seg in linear.default_split(k)):   # only whole groups of four scale blocks are all written
            plan = rng.choice(("fp4", "fp4_fp8"))
    else:
        m = _log_int(rng, 1, min(8192, 4 * 4096 * 4096 // k))
    return dict(op=op, m=m, n=n, k=k, plan=plan, norm=norm, bias=bias)


def _split(case):
    k = case["k"]
    return {"fp4": (k, 0, 0), "fp4_fp8": (k - 128, 0, 128)}.get(case["plan"]) or linear.default_split(k)


def _activations(g, m, k):
    x = torch.randn(m, k, generator=g, device=DEV)
    x[:, torch.randperm(k, generator=g, device=DEV)[:k // 32]] *= 30.0
    return x.to(torch.bfloat16)


def _weights(g, n, k):
    return (torch.randn(n, k, generator=g, device=DEV) * 0.02).to(torch.bfloat16)


def _normalised(x, gamma):
    """What a layer behind an RMSNorm is calibrated on."""
    f = x.float()
    return (f * torch.rsqrt(f.square().mean(1, keepdim=True) + EPS)).to(torch.bfloat16) * gamma


def _layer(g, x, n, split, norm, bias):
    """A packed layer calibrated on x[M, K]."""
    k = x.shape[1]
    gamma = (1.0 + 0.1 * torch.randn(k, generator=g, device=DEV)).to(torch.bfloat16) if norm else None
    index = abi.calibrate_reorder_index(_normalised(x, gamma) if norm else x)
    b = (0.1 * torch.randn(n, generator=g, device=DEV)).to(torch.bfloat16) if bias else None
    packed = linear.PackedWeights.from_float(_weights(g, n, k), index, split)
    return linear.MixedLinear(packed, bias=b, norm_weight=gamma, eps=EPS)


def _graph_shapes(case):
    """(N, K, norm) of one decoder layer's projections: qkv with a quarter of the heads for keys and for values,
    attention output, gate and up, down."""
    k, inner = case["k"], case["n"]
    return (k + k // 2, k, case["norm"]), (k, k, False), (2 * inner, k, case["norm"]), (k, inner, False)


def prepare(case, seed):
    g = torch.Generator(device=DEV).manual_seed(int(seed))
    op, m, n, k = case["op"], case["m"], case["n"], case["k"]
    split = _split(case)
    if op == "linear":
        x = _activations(g, m, k)
        # decode: m sequences of one token; above that one sequence of m tokens
        return op, _layer(g, x, n, split, case["norm"], case["bias"]), x.view(m, 1, k) if m <= 32 else x.view(1, m, k)
    if op == "graph":
        layers, inputs = [], []
        for ni, ki, norm in _graph_shapes(case):
            x = _activations(g, m, ki)
            layers.append(_layer(g, x, ni, linear.default_split(ki), norm, False))
            inputs.append(x.view(m, 1, ki))
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            for layer, x in zip(layers, inputs):
                layer(x)
        side.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            outputs = [layer(x) for layer, x in zip(layers, inputs)]
        return op, graph, outputs, layers, inputs
    if op == "module":
        x = _activations(g, m, k)
        index = abi.calibrate_reorder_index(x)
        module = _extension()
        return op, module, x, index, split, module.reorder_quantize_w(_weights(g, n, k), index, *split, n, k)
    if op == "pack":
        index = torch.randperm(k, generator=g, device=DEV).to(torch.int16)
        return op, _weights(g, n, k), index, split
    x = _activations(g, m, k)
    if op == "calibrate":
        return op, x
    out = abi.alloc_quant_outputs(m, *split, abi.MG_OPERAND_A, x.device)
    for t in out:
        t.zero_()   # scales of rows past the last one are never written
    return op, x, abi.calibrate_reorder_index(x), split, out


def _extension():
    """The extension module, from where the package's build puts it."""
    path = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(mixedgemm_amd.__file__))), "build")
    if path not in sys.path:
        sys.path.insert(0, path)
    return importlib.import_module("mixedgemm")


def run(state):
    op = state[0]
    if op == "linear":
        return state[1](state[2])
    if op == "graph":
        state[1].replay()
        return state[2]
    if op == "module":
        _, module, x, index, split, b = state
        a = module.reorder_quantize_x(x, index, *split, x.shape[0], b[0].shape[0])
        return module.matmul(a[0], b[0], a[1], b[1], a[2], b[2], a[3], b[3], a[4], b[4], a[5], b[5])
    if op == "pack":
        packed = linear.PackedWeights.from_float(*state[1:])
        return packed.tensors()
    if op == "calibrate":
        return torch.ops.mixedgemm_amd.calibrate_reorder_index(state[1])
    _, x, index, split, out = state
    return abi.reorder_quantize_x(x, index, *split, out=out)


def _linear_work(m, n, k, norm, bias):
    b = 2 * m * k + 2 * k + n * k // 2 + n * k // 32 + 2 * m * n + (2 * k if norm else 0) + (2 * n if bias else 0)
    return b, 2 * m * n * k


def work(case):
    op, m, n, k = case["op"], case["m"], case["n"], case["k"]
    kn, ks, ko = _split(case)
    if op == "graph":
        each = [_linear_work(m, ni, ki, norm, False) for ni, ki, norm in _graph_shapes(case)]
        return {"bytes": sum(b for b, _ in each), "flops": sum(f for _, f in each)}
    if op in ("linear", "module"):
        b, f = _linear_work(m, n, k, case["norm"], case["bias"])
        return {"bytes": b, "flops": f}
    if op == "pack":
        return {"bytes": 2 * n * k + 2 * k + n * k // 2 + n * k // 32, "flops": 0}
    if op == "calibrate":
        return {"bytes": 2 * m * k + 2 * k, "flops": 0}
    return {"bytes": m * (2 * k + kn // 2 + ks * 3 // 4 + ko + k // 32) + 2 * k, "flops": 0}


def tolerance(case):
    """Codes, scales and indices are bytes and whole numbers that the semantics fix. A GEMM's result is an fp32 sum
    rounded once to bf16: another order of summation moves a value by a bf16 step (2**-8 of it) now and then, and a
    sum that cancels by more, against the result's root mean square."""
    if case["op"] in ("quantize", "pack", "calibrate"):
        return "exact"
    return {"rel": 4e-3, "max": 1.6e-2}
