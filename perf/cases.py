"""The work a user of this library has it do, as cases that can be timed: the sparse linear over its whole range (one
decode step of a single projection up to prefill-sized B), the four chained linears of a decoder layer in both
directions of inference, and the compression of a weight on the GPU and on the host.

A case is a dict of plain values; "kind" says which public entry point it goes through:
  linear    spmm_splitk on a weight that is resident on the GPU (SpMM_SplitK_API)
  layer     DecoderLayer.forward (flashllm_decoder_layer_linears)
  compress  device_compress of a dense device-resident matrix (flashllm_device_tile_offsets / _compress)
  load      SparseWeight of a dense host matrix (InitSparseMatrixA_API[_NoReorder] and the copy to the GPU)
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.abspath("flash-llm_amd"))  # the package's folder is no importable name
import flashllm_spmm as F  # noqa: E402

MAX_WEIGHT = 49152 * 12288           # elements of the largest weight, also for drawn cases
MAX_MACS = 12 * 7168 * 7168 * 512    # multiply-adds of the largest case, also for drawn cases
MAX_COMPRESS = 27648 * 9216          # elements of the largest matrix compressed on the GPU
MAX_LOAD = 7168 * 7168               # ... and on the host


def _linear(name, m, k, n, sparsity, rows=False, split_k=0):
    return {"name": name, "kind": "linear", "m": m, "k": k, "n": n, "sparsity": sparsity, "rows": rows, "split_k": split_k}


def listed():
    return [
        # a small projection for one batch of eight sequences: latency, launches and the call itself
        _linear("linear-1024x1024-n8", 1024, 1024, 8, 0.8),
        # the smallest weight of the benchmark grid (attention output, hidden 7168), an ordinary decode step
        _linear("linear-7168x7168-n16", 7168, 7168, 16, 0.8),
        # odd numbers of row tiles (37) and k tiles (81), lower sparsity, a Split_K of the caller's own choice
        _linear("linear-4736x5184-n32-split4", 4736, 5184, 32, 0.7, split_k=4),
        # the benchmark workload: ffn up-projection, hidden 9216, 16 tokens, 80 %
        _linear("linear-36864x9216-n16", 36864, 9216, 16, 0.8),
        # ffn down-projection (long K, few rows) at the largest decode batch and the highest sparsity
        _linear("linear-9216x36864-n64-s90", 9216, 36864, 64, 0.9),
        # the largest weight of the grid, rows of very different density
        _linear("linear-49152x12288-n32-rows", 49152, 12288, 32, 0.8, rows=True),
        # B wider than a decode batch: speculative or chunked decoding
        _linear("linear-36864x9216-n128", 36864, 9216, 128, 0.8),
        # an odd multiple of 128 columns: a short prefill chunk
        _linear("linear-21504x7168-n384", 21504, 7168, 384, 0.8),
        # one decode step of a whole layer's linears
        {"name": "layer-9216-t16", "kind": "layer", "hidden": 9216, "tokens": 16, "sparsity": 0.8},
        # the same for a prefill chunk of 512 tokens (where the layer's linears run with Split_K = 1)
        {"name": "layer-7168-t512", "kind": "layer", "hidden": 7168, "tokens": 512, "sparsity": 0.8},
        # a weight pruned in device memory is compressed there (QKV, hidden 9216)
        {"name": "compress-27648x9216", "kind": "compress", "m": 27648, "k": 9216, "sparsity": 0.8},
        # a weight read from a checkpoint is compressed on the host and sent to the GPU
        {"name": "load-7168x7168", "kind": "load", "m": 7168, "k": 7168, "sparsity": 0.8, "reorder": True},
    ]


def _spread(rng, lo, hi):
    """A whole number from lo to hi, spread evenly over the logarithm."""
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def _shape(rng, limit):
    while True:
        m, k = 128 * _spread(rng, 8, 384), 64 * _spread(rng, 16, 768)
        if m * k <= limit:
            return m, k


def draw(rng):
    kind = rng.choices(["linear", "layer", "compress", "load"], [12, 3, 2, 1])[0]
    sparsity = round(rng.uniform(0.7, 0.9), 3)
    if kind == "linear":
        while True:
            m, k = _shape(rng, MAX_WEIGHT)
            n = rng.choice([8, 16, 32, 64]) if rng.random() < 0.7 else 128 * rng.randint(1, 5)
            if m * k * n <= MAX_MACS:
                break
        split_k = min(rng.choice([1, 2, 4, 8]), k // 64) if rng.random() < 0.25 else 0
        return {"kind": kind, "m": m, "k": k, "n": n, "sparsity": sparsity, "rows": rng.random() < 0.25, "split_k": split_k}
    if kind == "layer":
        while True:
            hidden = 128 * _spread(rng, 8, 72)
            tokens = rng.choice([8, 16, 32, 64]) if rng.random() < 0.6 else 128 * rng.randint(1, 4)
            if 12 * hidden * hidden * tokens <= MAX_MACS:
                return {"kind": kind, "hidden": hidden, "tokens": tokens, "sparsity": sparsity}
    m, k = _shape(rng, MAX_COMPRESS if kind == "compress" else MAX_LOAD)
    case = {"kind": kind, "m": m, "k": k, "sparsity": sparsity}
    if kind == "load":
        case["reorder"] = rng.random() < 0.5
    return case


# ---- inputs ---------------------------------------------------------------------------------------------------


def _pruned(m, k, sparsity, rows, gen):
    """Dense fp16 weights ~ N(0, 0.02) with an unstructured keep-mask; rows: the keep probability of a row is
    Beta(2, 8) distributed (the second smallest of nine uniforms), scaled to the wanted mean."""
    keep = 1.0 - sparsity
    if rows:
        p = torch.sort(torch.rand(m, 9, device="cuda", generator=gen), dim=1).values[:, 1:2]
        keep = torch.clamp(p * (keep / p.mean()), 0.0, 1.0)
    a = torch.empty(m, k, dtype=torch.float16, device="cuda")
    step = max(1, (1 << 27) // k)
    for r in range(0, m, step):
        block = a[r:r + step]
        block.normal_(0.0, 0.02, generator=gen)
        kept = keep[r:r + step] if rows else keep
        block.masked_fill_(torch.rand(block.shape, device="cuda", generator=gen) >= kept, 0.0)
    return a


def _with_fixed_size(a, sparsity, gen):
    """A few more weights kept (about six standard deviations of the number of nonzeros, under 0.1 % of them), four at
    a time in one row of a tile, so that the compressed size is the same whatever the seed."""
    m, k = a.shape
    t = a.view(m // 128, 128, k // 64, 64)
    tiles = (m // 128) * (k // 64)
    vectors = int(((t != 0).sum((1, 3)) + 3).div(4, rounding_mode="floor").sum())
    wanted = math.ceil((m * k * (1.0 - sparsity) + 1.5 * tiles + 6.0 * math.sqrt(m * k * sparsity * (1.0 - sparsity))) / 4)
    assert wanted >= vectors
    j = torch.arange(wanted - vectors, device="cuda")
    at = (j % tiles // (k // 64), j // tiles, j % tiles % (k // 64))  # one (row tile, row, k tile) each
    lines = t[at]
    zeros = torch.topk((lines == 0).to(torch.int8), 4, dim=1).indices
    sign = torch.randint(0, 2, zeros.shape, device="cuda", generator=gen).to(a.dtype) * 2 - 1
    t[at] = lines.scatter(1, zeros, 0.02 * sign)
    return a


class _Weight:
    """A weight compressed on the GPU, with what DecoderLayer asks of one."""

    def __init__(self, m, k, sparsity, rows, gen):
        self.m, self.k, self.split_k = m, k, None
        self.comp, self.offs = F.device_compress(_pruned(m, k, sparsity, rows, gen))

    def as_struct(self):
        return F.SparseWeightStruct(self.comp.data_ptr(), self.offs.data_ptr(), self.m, self.k, 0)


def _halfs(n):
    return torch.empty(n, dtype=torch.float16, device="cuda")


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    kind = case["kind"]
    if kind == "linear":
        m, k, n = case["m"], case["k"], case["n"]
        w = _Weight(m, k, case["sparsity"], case["rows"], gen)
        split_k = case["split_k"] or F.splitk_heuristic(m, n, k)
        return {"kind": kind, "w": w, "b": _halfs(n * k).normal_(generator=gen), "c": _halfs(n * m), "n": n,
                "split_k": split_k, "workspace": _halfs(split_k * n * m)}
    if kind == "layer":
        h, tokens = case["hidden"], case["tokens"]
        weights = [_Weight(m, k, case["sparsity"], False, gen) for m, k in ((3 * h, h), (h, h), (4 * h, h), (h, 4 * h))]
        layer = F.DecoderLayer(*weights)
        return {"kind": kind, "layer": layer, "x": _halfs(h * tokens).normal_(generator=gen), "tokens": tokens,
                "buffers": [_halfs(r * tokens) for r in (3 * h, h, h, 4 * h, h)],
                "workspace": _halfs(layer.workspace_halfs(tokens))}
    a = _with_fixed_size(_pruned(case["m"], case["k"], case["sparsity"], False, gen), case["sparsity"], gen)
    if kind == "compress":
        return {"kind": kind, "a": a}
    return {"kind": kind, "a": a.cpu().numpy(), "reorder": case["reorder"]}


def run(state):
    kind = state["kind"]
    if kind == "linear":
        w = state["w"]
        F.spmm_splitk(w.comp, w.offs, state["b"], state["c"], w.m, state["n"], w.k, state["workspace"], state["split_k"])
        return state["c"]
    if kind == "layer":
        _, (qkv, _, attn_out, ffn_mid, y) = state["layer"].forward(state["x"], state["tokens"], buffers=state["buffers"],
                                                                   workspace=state["workspace"])
        return {"qkv": qkv, "attn_out": attn_out, "ffn_mid": ffn_mid, "y": y}
    if kind == "compress":
        return F.device_compress(state["a"])
    w = F.SparseWeight(state["a"], reorder=state["reorder"])
    return w.comp, w.offs


# ---- what a pass cannot do without -------------------------------------------------------------------------------


def _compressed_bytes(m, k, sparsity):
    """Compressed_A (a 4-byte item per nonzero, tiles padded to four items: 1.5 on average) and TileOffsets."""
    tiles = (m // 128) * (k // 64)
    return 4 * (m * k * (1.0 - sparsity) + 1.5 * tiles) + 4 * (tiles + 2)


def work(case):
    """bytes: weights, B and C once.  flops: those of the dense product, as the method computes as dense."""
    kind = case["kind"]
    if kind == "linear":
        m, k, n = case["m"], case["k"], case["n"]
        return {"bytes": _compressed_bytes(m, k, case["sparsity"]) + 2 * k * n + 2 * m * n, "flops": 2.0 * m * k * n}
    if kind == "layer":
        h, t = case["hidden"], case["tokens"]
        return {"bytes": _compressed_bytes(12 * h, h, case["sparsity"]) + 2 * h * t * (1 + 3 + 1 + 4 + 1), "flops": 24.0 * h * h * t}
    m, k = case["m"], case["k"]
    return {"bytes": 2 * m * k + _compressed_bytes(m, k, case["sparsity"]), "flops": 0}


def tolerance(case):
    """fp16 in and out, fp32 sums, fp16 partial sums between the Split_K slices.  Measured against a product in 64 bits:
    rel 2.1e-4 (Split_K = 1) to 3.1e-4, two values of Split_K against each other up to 4.2e-4, largest single difference
    2.3e-3; over the four linears of a layer up to 5.9e-4 and 3.4e-3.  Stated: about four times what two correct
    implementations differ by.  The compressors produce defined bytes."""
    if case["kind"] == "linear":
        return {"rel": 1.6e-3, "max": 1e-2}
    if case["kind"] == "layer":
        return {"rel": 3e-3, "max": 2e-2}
    return "exact"
