"""The work that a program using this framework has it do, as measured cases.

Four kinds of case, all through the public entry points:

* ``layer``: one W4A4 layer step of ``my_int4.chain.make_chain`` (fused WUSH
  transform + quantization of bf16 activations, then the group-scaled product
  with INT4 weights), called eagerly, at decode, small-batch and prefill M;
* ``stack``: a decode step over several such layers, captured once with
  ``my_int4.chain.graphed`` and replayed, each layer with weights of its own;
* ``quant``: offline weight quantization, ``_C.quant_int4``;
* ``tensor``: the per-tensor-scale route, ``_C.quant_int4_tensor_scale_dev``
  followed by ``_C.w4a4_gemm_cutlass_dev``.

Inputs are made from the seed alone, in plain torch: bf16 activations N(0, 1)
with 1% outlier channels (x50), well-conditioned 32x32 transform blocks, and
N(0, 0.02) weights already in INT4 codes and bf16 scales, which is what an
inference program loads.
"""
import math

import torch

from my_int4 import _C
from my_int4.chain import graphed, make_chain

DEV = "cuda"
GROUP = 32
CLIP = 0.35337862372398376      # sigma-clip: largest code at 2.473650 sigma
LARGEST = 4096 * 57344 * 8192   # M * N * K of the largest case


def listed():
    return [
        # one token of one user, a small square projection: launches and latency
        {"name": "decode 1x4096x4096", "kind": "layer", "M": 1, "N": 4096, "K": 4096},
        # one token through a 70B feed-forward layer: the weight stream
        {"name": "decode 1x57344x8192", "kind": "layer", "M": 1, "N": 57344, "K": 8192},
        # eight users' tokens through a captured stack of feed-forward layers
        {"name": "stack 8x24576x4096", "kind": "stack", "M": 8, "N": 24576, "K": 4096, "layers": 4},
        # a ragged small batch
        {"name": "batch 13x24576x4096", "kind": "layer", "M": 13, "N": 24576, "K": 4096},
        # continuous batching, 70B feed-forward
        {"name": "batch 32x57344x8192", "kind": "layer", "M": 32, "N": 57344, "K": 8192},
        # larger batch through a down projection: long K, few columns
        {"name": "batch 64x4096x12288", "kind": "layer", "M": 64, "N": 4096, "K": 12288},
        # a short prompt of odd length, square projection
        {"name": "prompt 203x8192x8192", "kind": "layer", "M": 203, "N": 8192, "K": 8192},
        # a chunk of prefill with a ragged number of rows, down projection
        {"name": "prefill 1000x4096x12288", "kind": "layer", "M": 1000, "N": 4096, "K": 12288},
        # ordinary prefill, square projection
        {"name": "prefill 2048x4096x4096", "kind": "layer", "M": 2048, "N": 4096, "K": 4096},
        # the largest: long-prompt prefill of a 70B feed-forward layer
        {"name": "prefill 4096x57344x8192", "kind": "layer", "M": 4096, "N": 57344, "K": 8192},
        # loading a model: quantizing one bf16 weight matrix
        {"name": "quantize 24576x4096", "kind": "quant", "N": 24576, "K": 4096, "dtype": "bf16"},
        # the per-tensor-scale route at a prefill chunk
        {"name": "tensor 512x24576x4096", "kind": "tensor", "M": 512, "N": 24576, "K": 4096},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: any M up to the largest prefill, widths of 512 to 57344
    columns (odd ones among them), K a multiple of 256 as in most models or,
    one time in four, of 64 only."""
    kind = rng.choice(["layer"] * 7 + ["stack", "quant", "tensor"])
    step = 64 if rng.random() < 0.25 else 256
    K = max(step, _log(rng, 1024, 16384) // step * step)
    N = _log(rng, 512, 57344)
    if rng.random() < 0.7:
        N = (N + 63) // 64 * 64
    N = min(N, 57344 * 8192 // K)
    if kind == "quant":
        return {"kind": kind, "N": N, "K": K, "dtype": rng.choice(["bf16", "bf16", "fp16", "fp32"])}
    if kind == "stack":
        return {"kind": kind, "M": rng.randint(1, 8), "N": N, "K": K, "layers": 4}
    M = min(_log(rng, 1, 4096), LARGEST // (N * K))
    return {"kind": kind, "M": M, "N": N, "K": K}


# ------------------------------------------------------------------- inputs
def _generator(seed, salt):
    return torch.Generator(device=DEV).manual_seed(seed * 1000003 + salt)


def _activations(g, M, K):
    x = torch.randn(M, K, generator=g, device=DEV)
    hot = torch.randperm(K, generator=g, device=DEV)[: max(1, K // 100)]
    x[:, hot] *= 50.0
    return x.to(torch.bfloat16)


def _transform(seed, K):
    """(K/32, 32, 32) blocks: an orthogonal matrix with its inputs scaled."""
    g = torch.Generator().manual_seed(seed * 1000003 + 7)
    C = K // GROUP
    q = torch.linalg.qr(torch.randn(C, GROUP, GROUP, generator=g))[0]
    scale = torch.exp(0.3 * torch.randn(C, 1, GROUP, generator=g))
    return (q * scale).to(torch.bfloat16).contiguous().to(DEV)


def _codes(x):
    """sigma-clip codes (integers as floats) and scales of (..., 32) groups."""
    mean = x.mean(-1, keepdim=True)
    var = (x * x).mean(-1, keepdim=True) - mean * mean
    s = (var.clamp_min(0).sqrt() * CLIP + 1e-8).to(torch.bfloat16)
    return (x / s.to(x.dtype)).round().clamp(-7, 7), s.squeeze(-1)


def _pack(q):
    """(rows, K) integer codes -> two codes per byte, the even one low."""
    u = q.to(torch.int32) & 15
    return (u[:, 0::2] | (u[:, 1::2] << 4)).to(torch.uint8)


def _unpack(b):
    """The codes of _pack, in 64 bits."""
    u = torch.stack((b & 15, b >> 4), dim=-1).reshape(b.shape[0], -1).to(torch.float64)
    return torch.where(u > 7, u - 16, u)


def _weights(g, N, K):
    wq = torch.empty(N, K // 2, dtype=torch.uint8, device=DEV)
    ws = torch.empty(N, K // GROUP, dtype=torch.bfloat16, device=DEV)
    for n in range(0, N, 8192):
        w = torch.randn(min(8192, N - n), K // GROUP, GROUP, generator=g, device=DEV) * 0.02
        q, s = _codes(w)
        wq[n:n + 8192] = _pack(q.reshape(q.shape[0], K))
        ws[n:n + 8192] = s
    return wq, ws


def _layer_inputs(case, seed, layer=0):
    M, N, K = case["M"], case["N"], case["K"]
    g = _generator(seed, 11 + 100 * layer)
    return (_activations(g, M, K), _transform(seed + 7919 * layer, K)) + _weights(g, N, K)


def _quant_input(case, seed):
    dt = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}[case["dtype"]]
    w = torch.empty(case["N"], case["K"], dtype=dt, device=DEV)
    g = _generator(seed, 13)
    for n in range(0, case["N"], 8192):
        w[n:n + 8192] = torch.randn(min(8192, case["N"] - n), case["K"], generator=g, device=DEV) * 0.02
    return w


def _tensor_inputs(case, seed):
    g = _generator(seed, 17)
    M, N, K = case["M"], case["N"], case["K"]
    x = torch.randn(M, K, generator=g, device=DEV).to(torch.bfloat16)
    wq = torch.empty(N, K // 2, dtype=torch.uint8, device=DEV)
    for n in range(0, N, 8192):
        w = torch.randn(min(8192, N - n), K, generator=g, device=DEV)
        wq[n:n + 8192] = _pack((w / CLIP).round().clamp(-7, 7))
    inv = torch.tensor([1.0 / CLIP], device=DEV)            # codes of N(0, 1) activations
    alpha = torch.tensor([CLIP * CLIP * 0.02], device=DEV)  # both scales
    return x, wq, inv, alpha


# -------------------------------------------------------------------- cases
def prepare(case, seed):
    if case["kind"] == "layer":
        return {"kind": "layer", "step": make_chain(*_layer_inputs(case, seed))}
    if case["kind"] == "stack":
        steps = [make_chain(*_layer_inputs(case, seed, i)) for i in range(case["layers"])]
        graph, ys = graphed(lambda: [s() for s in steps])
        return {"kind": "stack", "graph": graph, "ys": ys, "steps": steps}
    if case["kind"] == "quant":
        return {"kind": "quant", "w": _quant_input(case, seed)}
    return {"kind": "tensor", "args": _tensor_inputs(case, seed)}


def run(state):
    if state["kind"] == "layer":
        return state["step"]()
    if state["kind"] == "stack":
        state["graph"].replay()
        return state["ys"]
    if state["kind"] == "quant":
        return _C.quant_int4(state["w"])
    x, wq, inv, alpha = state["args"]
    return _C.w4a4_gemm_cutlass_dev(_C.quant_int4_tensor_scale_dev(x, inv), wq, alpha)


def work(case):
    """Bytes: inputs read once, outputs written once; flops: the products."""
    N, K = case["N"], case["K"]
    weights = N * K / 2 + N * K / 16
    if case["kind"] == "quant":
        return {"bytes": N * K * (4 if case["dtype"] == "fp32" else 2) + weights, "flops": 0}
    M = case["M"]
    if case["kind"] == "tensor":
        return {"bytes": 2 * M * K + N * K / 2 + 2 * M * N, "flops": 2 * M * N * K}
    layers = case.get("layers", 1)
    return {"bytes": layers * (2 * M * K + 64 * K + weights + 2 * M * N),
            "flops": layers * (2 * M * N * K + 64 * M * K)}


def tolerance(case):
    """Codes, scales and the per-tensor product (exact integer sums, one
    rounding) are the same bits in every correct implementation.  The
    group-scaled product is summed in fp32 in any order and rounded once to
    fp16: 2.1e-4 to 2.9e-4 from the 64-bit product as measured; four times
    that, and four half units of fp16 for the largest difference."""
    if case["kind"] in ("quant", "tensor"):
        return "exact"
    return {"rel": 1e-3, "max": 2e-3}


# ------------------------------------------------------------ in 64 bits
def _exact_layer(x, t, wq, ws):
    M, K = x.shape
    C = K // GROUP
    xb = x.double().view(M, C, GROUP).transpose(0, 1).contiguous()
    xt = torch.bmm(xb, t.double().transpose(1, 2).contiguous()).transpose(0, 1).contiguous()
    q, s = _codes(xt)
    xd = (q * s.double().unsqueeze(-1)).view(M, K)
    N = wq.shape[0]
    y = torch.empty(M, N, dtype=torch.float64, device=DEV)
    for n in range(0, N, 8192):
        w = _unpack(wq[n:n + 8192]).view(-1, C, GROUP) * ws[n:n + 8192].double().unsqueeze(-1)
        y[:, n:n + 8192] = xd @ w.view(-1, K).t().contiguous()
    return y.view(N) if M == 1 else y


def exact(case, seed):
    if case["kind"] == "layer":
        return _exact_layer(*_layer_inputs(case, seed))
    if case["kind"] == "stack":
        return [_exact_layer(*_layer_inputs(case, seed, i)) for i in range(case["layers"])]
    if case["kind"] == "quant":
        w = _quant_input(case, seed)
        s = torch.empty(case["N"], case["K"] // GROUP, dtype=torch.float64, device=DEV)
        for n in range(0, case["N"], 8192):
            g = w[n:n + 8192].double().view(-1, case["K"] // GROUP, GROUP)
            mean = g.mean(-1)
            s[n:n + 8192] = ((g * g).mean(-1) - mean * mean).clamp_min(0).sqrt() * CLIP + 1e-8
        return [None, s]
    x, wq, inv, alpha = _tensor_inputs(case, seed)
    q = (x.float() * inv).round().clamp(-7, 7).double()
    y = torch.empty(case["M"], case["N"], dtype=torch.float64, device=DEV)
    for n in range(0, case["N"], 8192):
        y[:, n:n + 8192] = q @ _unpack(wq[n:n + 8192]).t().contiguous()
    return y * alpha.double()
