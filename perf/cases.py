"""The work this library is used for, as cases that a timing harness can prepare and run.

A case is a dict of plain values.  Three kinds, by ``op``:

* ``"layer"``: ``layers`` quantized linear layers of one shape (``m`` rows, ``k`` in-features, ``n`` out-features),
  called one after the other, each with its own weights, as the same projection of successive blocks is;
* ``"step"``: everything quantized that one step of a decoder-only network runs for ``m`` rows: per block the query,
  key, value and output projections (``hidden`` x ``hidden``), gate and up (``hidden`` -> ``ffn``) and down (``ffn`` ->
  ``hidden``), then the vocabulary projection (``hidden`` -> ``vocab``);
* ``"quantize"``: ``layers`` layers of that shape made from 16-bit weights, which is what loading a network does.

Quantization options in every case: ``bs`` block size, ``col`` blocks along K (else along N), ``zp`` with zero-points,
``dtype`` of activations, scales and weights before quantization, ``bias``.
Activations are drawn from N(0, 1) and weights from N(0, 0.02), as after a normalisation and after training.
"""

import math

import torch

import ms_blkq4linear_ext
from ms_blkq4linear import BlkQ4Linear


def _layer(name, m, n, k, layers, bs, col, zp, dtype, bias):
    return {"name": name, "op": "layer", "m": m, "n": n, "k": k, "layers": layers, "bs": bs, "col": col, "zp": zp,
            "dtype": dtype, "bias": bias}


def _step(name, m, hidden, ffn, vocab, blocks, bs, col, zp, dtype):
    return {"name": name, "op": "step", "m": m, "hidden": hidden, "ffn": ffn, "vocab": vocab, "blocks": blocks, "bs": bs,
            "col": col, "zp": zp, "dtype": dtype, "bias": False}


def _quantize(name, n, k, layers, bs, col, zp, dtype):
    return {"name": name, "op": "quantize", "n": n, "k": k, "layers": layers, "bs": bs, "col": col, "zp": zp,
            "dtype": dtype, "bias": False}


def listed():
    return [
        # one projection for one token: the smallest call there is, all latency
        _layer("one projection one token", 1, 4096, 4096, 1, 64, True, False, "float16", False),
        # one token of a conversation: every layer called once, weights from memory each time
        _step("decode step one token", 1, 4096, 11008, 128256, 2, 32, True, True, "float16"),
        # a dozen conversations decoded together in bfloat16
        _step("decode step 12 tokens bf16", 12, 4096, 11008, 128256, 2, 64, True, True, "bfloat16"),
        # the widest layer of a large network at batch 16
        _layer("batch 16 on a wide layer", 16, 28672, 8192, 3, 64, True, True, "float16", False),
        # a loaded server between decoding and prompts; biased up-projections
        _layer("batch 48 up-projection", 48, 11008, 4096, 8, 32, True, True, "float16", True),
        # weights quantized in blocks along N, an odd batch
        _layer("batch 150 blocks along N", 150, 4096, 4096, 8, 32, False, True, "float16", False),
        # a chunk of a prompt mixed with decoding
        _layer("chunk of 512", 512, 4096, 4096, 4, 64, True, True, "float16", True),
        # a prompt of no round length, bfloat16, without zero-points
        _layer("prompt of 777 bf16", 777, 11008, 4096, 2, 64, True, False, "bfloat16", False),
        # a prompt of 2048 tokens through one projection
        _layer("prompt of 2048", 2048, 4096, 4096, 1, 64, True, True, "float16", False),
        # the largest product: a batch of prompts through the widest layer, the finest blocks
        _layer("prompts of 4096 wide layer", 4096, 28672, 8192, 1, 16, True, True, "float16", False),
        # a network is loaded: the widest layer in the finest blocks
        _quantize("quantize a wide layer", 28672, 8192, 1, 16, True, True, "float16"),
        # and several ordinary layers in bfloat16, blocks along N
        _quantize("quantize bf16 along N", 11008, 4096, 4, 32, False, True, "bfloat16"),
    ]


def _log_uniform(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _options(rng):
    return {"bs": rng.choice((16, 32, 32, 64, 64, 64)), "col": rng.random() < 0.8, "zp": rng.random() < 0.7,
            "dtype": rng.choice(("float16", "float16", "bfloat16")), "bias": rng.random() < 0.25}


def draw(rng):
    """A case of the ranges above: 1 to 4096 rows, layers of 1024 to 28672 features either way (any multiple of 64)."""
    o = _options(rng)
    # a power of two or any multiple of 64 in between
    feature = lambda lo, hi: 64 * round(_log_uniform(rng, lo, hi) / 64)  # noqa: E731
    kind = rng.random()
    if kind < 0.15:
        hidden = 512 * rng.randint(4, 10)
        return {"op": "step", "m": round(_log_uniform(rng, 1, 64)), "hidden": hidden,
                "ffn": 64 * round(hidden * rng.uniform(2.5, 4.0) / 64), "vocab": 256 * rng.randint(125, 501), "blocks": 1,
                **o, "bias": False}
    if kind < 0.35:
        return {"op": "quantize", "n": feature(1024, 28672), "k": feature(1024, 8192), "layers": rng.randint(1, 2), **o,
                "bias": False}
    while True:
        m, n, k = round(_log_uniform(rng, 1, 4096)), feature(1024, 28672), feature(1024, 16384)
        if rng.random() < 0.3:
            m = max(1, 1 << round(math.log2(m)))
        if m * n * k <= 2048 * 28672 * 8192 and m * k <= 4096 * 8192:
            break
    layers = max(1, min(8, round(4096 * 28672 * 8192 / (64.0 * m * n * k))))
    layers = max(1, min(layers, 1500000000 // (n * k)))
    return {"op": "layer", "m": m, "n": n, "k": k, "layers": layers, **o}


def _dtype(case):
    return getattr(torch, case["dtype"])


def _calls(case):
    """(rows, in-features, out-features, which input) of every layer that one pass calls, in order."""
    if case["op"] == "step":
        h, f = case["hidden"], case["ffn"]
        block = [(h, h, 0), (h, h, 0), (h, h, 0), (h, h, 1), (h, f, 0), (h, f, 0), (f, h, 2)]
        shapes = block * case["blocks"] + [(h, case["vocab"], 1)]
    else:
        shapes = [(case["k"], case["n"], i) for i in range(case["layers"])]
    return [(case.get("m", 0), k, n, i) for k, n, i in shapes]


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)

    def normal(*shape, scale=1.0):
        return torch.randn(*shape, generator=gen, device="cuda", dtype=_dtype(case)).mul_(scale)

    if case["op"] == "quantize":
        return {"case": case, "weights": [normal(n, k, scale=0.02) for _, k, n, _ in _calls(case)]}
    layers, inputs, which = [], {}, []
    for m, k, n, i in _calls(case):
        bias = normal(n, scale=0.1) if case["bias"] else None
        layers.append(BlkQ4Linear(case["bs"], case["col"], not case["zp"], normal(n, k, scale=0.02), bias))
        if i not in inputs:
            inputs[i] = normal(m, k)
        which.append(inputs[i])
    return {"case": case, "layers": layers, "inputs": which}


def run(state):
    case = state["case"]
    if case["op"] == "quantize":
        return [ms_blkq4linear_ext.quant(case["bs"], case["col"], case["zp"], w) for w in state["weights"]]
    return [layer(x) for layer, x in zip(state["layers"], state["inputs"])]


def work(case):
    total, flops = 0, 0
    for m, k, n, _ in _calls(case):
        blocks = k * n // case["bs"]
        packed = k * n // 2 + blocks * (3 if case["zp"] else 2)
        if case["op"] == "quantize":
            total += 2 * k * n + packed
            flops += 2 * k * n  # one multiply and one add per weight
        else:
            total += packed + 2 * m * k + 2 * m * n + (2 * n if case["bias"] else 0)
            flops += 2 * m * k * n
    return {"bytes": total, "flops": flops}


def tolerance(case):
    # Packed weights, scales and zero-points are defined bit for bit.  A product is rounded once to 16 bits from 32-bit
    # sums of once-rounded weights: against the same sums in 64 bits, not rounded, it differs by 2.1e-4 (float16) and
    # 1.7e-3 (bfloat16) in the 2-norm.  A bias is added to the rounded product and the sum rounded again: 2.95e-4 and
    # 2.4e-3.  Four times that.
    if case["op"] == "quantize":
        return "exact"
    return {"rel": {"float16": 8e-4, "bfloat16": 6.7e-3}[case["dtype"]] * (1.4 if case["bias"] else 1.0)}
