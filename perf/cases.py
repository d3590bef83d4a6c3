"""The workloads this repository's speed is judged on, each ONE call (or one decoder layer, or one generation)
through the public entry points of the ``sbvr`` package, over the range of sizes, plane counts, group lengths,
index widths and batch rows that its configurations, tests and benchmark use.

A case is a dict of plain values; ``kind`` names the entry point:

  linear    SBVRLinear.forward of M rows: x (M, K) -> (M, N)
  layer     the four SBVRLinear of one Llama-3-8B-shaped layer (q|k|v, o, gate|up, down) at M rows
  mm_T      sbvr.mm_T: both operands encoded
  online    sbvr.online_mm_T: activations encoded on the fly, then multiplied with the encoded weight
  row_deq   _sbvr_row_deq_mm_T: fp16 activations against a weight encoded with trans=True
  decode    sbvr.decode: the dense weight of an encoded one
  encode    sbvr.sbvr(W): encoding a weight
  generate  SbvrLlamaDecoder.generate: a prompt, then greedy tokens, batch 1

N output features, K input features, S bit planes, G group length, L lines of the coefficient table (more than
256: 16-bit indices)."""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "sbvr-cpu-arm_amd"))

import sbvr  # noqa: E402
from sbvr import synth  # noqa: E402
from sbvr.decoder import LlamaShape, SbvrLlamaDecoder  # noqa: E402

DEVICE = "cuda:0"
# the widths of a Llama-3-8B layer: rows of the fused q|k|v, hidden, feed-forward
QKV, HIDDEN, FFN = 6144, 4096, 14336


def listed():
    return [
        # one decoded token through the smallest projection (k or v): latency and the host path
        {"name": "kv-1", "kind": "linear", "M": 1, "N": 1024, "K": 4096, "S": 4, "G": 128, "L": 256, "bias": False},
        # one decoded token through a whole layer's linears: what an eager serving loop calls per layer
        {"name": "layer-1", "kind": "layer", "M": 1, "S": 4, "G": 128, "L": 256},
        # a dozen sequences decoded together through the down projection, three planes
        {"name": "down-12-s3", "kind": "linear", "M": 12, "N": 4096, "K": 14336, "S": 3, "G": 128, "L": 256, "bias": False},
        # a ragged prompt through the fused q|k|v with its three tables (16-bit indices), the reference's own group
        # length, and a bias
        {"name": "prompt-333-g256", "kind": "linear", "M": 333, "N": 6144, "K": 4096, "S": 4, "G": 256, "L": 768, "bias": True},
        # a prompt through a weight at the reference's highest quality (8 planes)
        {"name": "prompt-512-s8", "kind": "linear", "M": 512, "N": 4096, "K": 4096, "S": 8, "G": 256, "L": 256, "bias": False},
        # a 2048-token prompt through the 70B-width up projection: the largest
        {"name": "up70-2048", "kind": "linear", "M": 2048, "N": 28672, "K": 8192, "S": 4, "G": 128, "L": 256, "bias": False},
        # both operands encoded ahead of time, a few rows (the product the reference's kernels compute)
        {"name": "both-encoded-4", "kind": "mm_T", "M": 4, "N": 4096, "K": 4096, "Sl": 4, "S": 4, "G": 256, "L": 256},
        # sixteen rows of activations encoded on the fly with the default 8 input planes
        {"name": "online-16", "kind": "online", "M": 16, "N": 4096, "K": 4096, "Sl": 8, "S": 4, "G": 128, "L": 256},
        # a few rows against a weight encoded in the transposed layout
        {"name": "trans-3", "kind": "row_deq", "M": 3, "N": 4096, "K": 4096, "S": 4, "G": 256, "L": 256},
        # the dense weight back from an encoded gate projection
        {"name": "decode-gate", "kind": "decode", "N": 14336, "K": 4096, "S": 4, "G": 128, "L": 256},
        # encoding a k or v projection
        {"name": "encode-kv", "kind": "encode", "N": 1024, "K": 4096, "S": 4, "G": 128},
        # the 8B-shaped decoder: a 128-token prompt, then 128 greedy tokens
        {"name": "generate-8b", "kind": "generate", "layers": 32, "prompt": 128, "new": 128},
    ]


def _spread(rng, lo, hi):
    """An integer between lo and hi, spread over its logarithm."""
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def _size(rng, lo, hi, step):
    return step * _spread(rng, lo // step, hi // step)


def draw(rng):
    kind = rng.choice(["linear"] * 7 + ["layer", "mm_T", "online", "row_deq", "decode", "encode", "generate"])
    S = rng.choice([4, 4, 4, 2, 3, 6, 8])
    G = rng.choice([128, 128, 256, 256, 64])
    L = rng.choice([256, 256, 16, 300, 768])
    if kind == "linear":
        # (a third of the row counts below 32: the batches of decoding; the rest up to the longest prompt)
        M = _spread(rng, 1, 32) if rng.random() < 0.34 else _spread(rng, 1, 2048)
        N, K = _spread(rng, 512, 28672), _size(rng, 512, 28672, 256)
        while N * K > 8192 * 28672:
            N, K = _spread(rng, 512, 28672), _size(rng, 512, 28672, 256)
        return {"kind": kind, "M": M, "N": N, "K": K, "S": S, "G": G, "L": L, "bias": rng.random() < 0.3}
    if kind == "layer":
        return {"kind": kind, "M": _spread(rng, 1, 64), "S": rng.choice([2, 3, 4]), "G": rng.choice([128, 256]), "L": L}
    if kind == "mm_T":
        return {"kind": kind, "M": _spread(rng, 1, 64), "N": _spread(rng, 512, 14336), "K": _size(rng, 512, 14336, 256),
                "Sl": rng.choice([4, 4, 2, 8]), "S": rng.choice([4, 4, 2, 3, 8]), "G": rng.choice([128, 256]), "L": L}
    if kind == "online":
        return {"kind": kind, "M": _spread(rng, 1, 64), "N": _spread(rng, 512, 14336), "K": _size(rng, 512, 14336, 256),
                "Sl": rng.choice([8, 8, 4]), "S": rng.choice([4, 4, 2, 3]), "G": rng.choice([128, 256]), "L": L}
    if kind == "row_deq":
        return {"kind": kind, "M": _spread(rng, 1, 32), "N": _size(rng, 512, 14336, 256), "K": _spread(rng, 512, 14336),
                "S": rng.choice([4, 4, 2, 3]), "G": rng.choice([128, 256]), "L": L}
    if kind == "decode":
        return {"kind": kind, "N": _spread(rng, 512, 14336), "K": _size(rng, 512, 8192, 256), "S": S, "G": G, "L": L}
    if kind == "encode":
        return {"kind": kind, "N": _spread(rng, 64, 1024), "K": _size(rng, 512, 4096, 256), "S": rng.choice([4, 3, 2]),
                "G": rng.choice([128, 256])}
    return {"kind": kind, "layers": _spread(rng, 2, 32), "prompt": _spread(rng, 1, 128), "new": _spread(rng, 1, 128)}


# -- inputs -----------------------------------------------------------------------------------------------

def _encoding(gen, rows, cols, S, G, L, sigma=0.02):
    """A random encoded weight (rows, cols), drawn on the device: Bernoulli(1/2) planes, uniform line indices and a
    table of lines shaped like the encoder's."""
    bvr = torch.randint(-2 ** 31, 2 ** 31, (cols // 32, rows, S), dtype=torch.int32, generator=gen,
                        device=DEVICE).view(torch.uint32)
    idx = torch.randint(0, L, (cols // G, rows), dtype=torch.int32, generator=gen, device=DEVICE)
    idx = idx.to(torch.uint8 if L <= 256 else torch.uint16)
    return bvr, idx, synth.make_lines(L, S, sigma, gen.initial_seed() % (1 << 31)).to(DEVICE)


def _activations(gen, *shape):
    return torch.randn(shape, generator=gen, device=DEVICE).to(torch.float16)


def _linear(gen, N, K, S, G, L, bias=False):
    bias = (torch.randn(N, generator=gen, device=DEVICE) * 0.1).to(torch.float16) if bias else None
    return sbvr.SBVRLinear(K, N, *_encoding(gen, N, K, S, G, L), G, bias)


def prepare(case, seed):
    c, gen = case, torch.Generator(device=DEVICE).manual_seed(seed)
    kind = c["kind"]
    if kind == "linear":
        return {"kind": kind, "linear": _linear(gen, c["N"], c["K"], c["S"], c["G"], c["L"], c["bias"]),
                "x": _activations(gen, c["M"], c["K"])}
    if kind == "layer":
        S, G, L, M = c["S"], c["G"], c["L"], c["M"]
        # (the fused matrices hold one table per weight that went into them)
        shapes = [(QKV, HIDDEN, 3 * L), (HIDDEN, HIDDEN, L), (2 * FFN, HIDDEN, 2 * L), (HIDDEN, FFN, L)]
        return {"kind": kind, "pairs": [(_linear(gen, n, k, S, G, lines), _activations(gen, M, k)) for n, k, lines in shapes]}
    if kind == "mm_T":
        lhs = sbvr.sbvr.from_parts(*_encoding(gen, c["M"], c["K"], c["Sl"], c["G"], 16, 1.0), c["G"])
        rhs = sbvr.sbvr.from_parts(*_encoding(gen, c["N"], c["K"], c["S"], c["G"], c["L"]), c["G"])
        return {"kind": kind, "lhs": lhs, "rhs": rhs}
    if kind == "online":
        enc = sbvr.sbvr.from_parts(*_encoding(gen, c["N"], c["K"], c["S"], c["G"], c["L"]), c["G"])
        # one line of input coefficients per group of K, as profile_input leaves them
        enc.input_num_sums = c["Sl"]
        lines = synth.make_lines(c["K"] // c["G"], c["Sl"], 1.0, seed % (1 << 31)).to(DEVICE)
        enc.input_coeff = torch.nn.Parameter(lines, requires_grad=False)
        return {"kind": kind, "enc": enc, "x": _activations(gen, c["M"], c["K"])}
    if kind == "row_deq":
        # (the encoded tensor is the transposed weight: K rows, groups along N)
        bvr, idx, cache = _encoding(gen, c["K"], c["N"], c["S"], c["G"], c["L"])
        return {"kind": kind, "w": (bvr, idx, cache), "x": _activations(gen, c["M"], c["K"]),
                "none": torch.zeros(0, dtype=torch.float16, device=DEVICE)}
    if kind == "decode":
        return {"kind": kind, "enc": sbvr.sbvr.from_parts(*_encoding(gen, c["N"], c["K"], c["S"], c["G"], c["L"]), c["G"])}
    if kind == "encode":
        return {"kind": kind, "w": torch.randn((c["N"], c["K"]), generator=gen, device=DEVICE) * 0.02,
                "config": {"num_sums": c["S"], "bvr_len": c["G"]}}
    dec = SbvrLlamaDecoder(LlamaShape(layers=c["layers"]), DEVICE, max_seq=256, seed=seed % (1 << 24))
    dec.capture()
    prompt = torch.randint(0, dec.shape.vocab, (c["prompt"],), generator=gen, device=DEVICE)
    return {"kind": kind, "decoder": dec, "prompt": prompt, "new": c["new"]}


# -- one pass ---------------------------------------------------------------------------------------------

def run(state):
    s, kind = state, state["kind"]
    if kind == "linear":
        return s["linear"](s["x"])
    if kind == "layer":
        return [linear(x) for linear, x in s["pairs"]]
    if kind == "mm_T":
        return sbvr.mm_T(s["lhs"], s["rhs"], None)
    if kind == "online":
        return s["enc"].online_mm_T(s["x"])
    if kind == "row_deq":
        return sbvr._sbvr_row_deq_mm_T(s["x"], *s["w"], s["none"])
    if kind == "decode":
        return s["enc"].decode()
    if kind == "encode":
        enc = sbvr.sbvr(s["w"], encoder_config=dict(s["config"]), device=DEVICE, verbose_level=0)
        # (how many lines the table ends up with, and with it the width of the indices, depends on the data: both are
        # returned in one shape for all data; at most one line per group)
        cache, idx = enc.coeff_cache.data, enc.coeff_idx.data
        cache = torch.nn.functional.pad(cache, (0, 0, 0, idx.numel() - cache.shape[0]))
        return {"bvr": enc.bvr.data.view(torch.int32), "cache": cache, "idx": idx.to(torch.int32)}
    tokens, _ = s["decoder"].generate(s["prompt"], s["new"])
    return {"tokens": tokens, "logits": s["decoder"].logits}


# -- what a pass cannot do without ------------------------------------------------------------------------

def _weight_bytes(rows, cols, S, G, L):
    return rows * cols * S / 8 + (cols // G) * rows * (1 if L <= 256 else 2) + 2 * L * S


def _linear_work(M, N, K, S, G, L):
    return _weight_bytes(N, K, S, G, L) + 2 * M * K + 2 * M * N, 2 * M * N * K


def work(case):
    c, kind = case, case["kind"]
    if kind in ("linear", "row_deq"):
        rows, cols = (c["N"], c["K"]) if kind == "linear" else (c["K"], c["N"])
        return {"bytes": _weight_bytes(rows, cols, c["S"], c["G"], c["L"]) + 2 * c["M"] * (c["K"] + c["N"]),
                "flops": 2 * c["M"] * c["N"] * c["K"]}
    if kind == "layer":
        parts = [_linear_work(c["M"], n, k, c["S"], c["G"], lines * c["L"])
                 for n, k, lines in ((QKV, HIDDEN, 3), (HIDDEN, HIDDEN, 1), (2 * FFN, HIDDEN, 2), (HIDDEN, FFN, 1))]
        return {"bytes": sum(b for b, _ in parts), "flops": sum(f for _, f in parts)}
    if kind in ("mm_T", "online"):
        left = 2 * c["M"] * c["K"] if kind == "online" else _weight_bytes(c["M"], c["K"], c["Sl"], c["G"], 16)
        return {"bytes": _weight_bytes(c["N"], c["K"], c["S"], c["G"], c["L"]) + left + 2 * c["M"] * c["N"],
                "flops": 2 * c["M"] * c["N"] * c["K"]}
    if kind == "decode":
        return {"bytes": _weight_bytes(c["N"], c["K"], c["S"], c["G"], c["L"]) + 2 * c["N"] * c["K"], "flops": 0}
    if kind == "encode":
        # every value against the points of one line at least: a difference, a square and a minimum each
        return {"bytes": 4 * c["N"] * c["K"] + _weight_bytes(c["N"], c["K"], c["S"], c["G"], 256),
                "flops": 3 * c["N"] * c["K"] * 2 ** c["S"]}
    s = LlamaShape(layers=c["layers"])
    per_layer = [(QKV, HIDDEN, 768), (HIDDEN, HIDDEN, 256), (2 * FFN, HIDDEN, 512), (HIDDEN, FFN, 256)]
    weights = s.layers * sum(_weight_bytes(n, k, 4, 128, lines) for n, k, lines in per_layer)
    head = 2 * s.vocab * s.hidden
    params = s.layers * sum(n * k for n, k, _ in per_layer)
    # the prompt in one pass over the weights, then one pass per new token
    return {"bytes": (c["new"] + 1) * (weights + head),
            "flops": 2 * params * (c["prompt"] + c["new"]) + (c["new"] + 1) * head}


def tolerance(case):
    """About four times what the paths differ by from the same products in 64 bits, over these ranges."""
    kind = case["kind"]
    if kind == "decode":
        return {"rel": 1e-5, "max": 2e-3}       # one rounding of an (almost always exact) 32-bit sum of S terms
    if kind == "encode":
        return "exact"
    if kind == "generate":
        # two orders of the same 32-bit sums, 32 layers deep: the logits 9e-3 apart
        return {"rel": 2e-2, "max": 0.2, "differ": 0.01}
    # fp16 results of 32-bit sums (2.1e-4), of weights rounded to fp16 once (3.5e-4) or plane by plane (4e-4)
    return {"rel": 1.6e-3 if case["S"] > 4 else 1e-3, "max": 8e-3}
