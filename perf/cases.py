"""The work a user of this framework has it do, as cases that can be timed.

Four kinds of pass, each through the public entry points of the package:

  amm      Amm.run_ptr on device tensors: closest-centroid search, table gather, de-quantisation.  int8 tables with
           one scale (`scale_group` 0) or one per codebook (1), or fp32 tables; `chain` runs a second operator of the
           transposed shape on an input of its own, as the two feed-forward matrices of an encoder layer follow each other.
  host     Amm.run on pageable numpy buffers in and out, what the C++ layer's amm_host hands over.
  forward  Transformer.forward on device features, launched op by op, or a replay of Transformer.capture's graph.
  lutgen   Context.lutgen: the offline construction and quantisation of a table from centroids and a dense weight.

Weights are random: centroids and activations N(0, 1), dense weights N(0, 0.02), tables = centroids x weight quantised
by its largest entry, which is what the converter does with a calibrated model.
"""
import math
import os
import sys

import numpy as np
import torch

ROOT = os.getcwd()
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)
from __graft_entry__ import load_package  # noqa: E402

_package = load_package()
_context = None


def _ctx():
    """One context for the process, on torch's stream, as a serving program holds it."""
    global _context
    if _context is None:
        _context = _package.Context(torch.cuda.current_device())
        _context.set_stream(torch.cuda.current_stream().cuda_stream)
    return _context


def _amm(name, n, k, v, c, m, lut="i8", scale_group=0, chain=False):
    return {"name": name, "kind": "amm", "n": n, "k": k, "v": v, "c": c, "m": m, "lut": lut, "scale_group": scale_group, "chain": chain}


def listed():
    return [
        # one token through a feed-forward matrix: nothing but launches and latency
        _amm("amm_one_token", 1, 768, 4, 16, 3072),
        # the single operator that the reference's CPU path can run: one short sentence
        _amm("amm_128_tokens", 128, 768, 2, 16, 768),
        # the two feed-forward matrices of BERT-base at 64 x 128 tokens: what bench.py times
        _amm("ffn_pair", 8192, 768, 4, 16, 3072, chain=True),
        # the reference's own tile-search operator at its full batch of 64 x 512 tokens
        _amm("amm_32768_tokens", 32768, 1024, 4, 16, 4096),
        # ViT-Base/16, 64 images of 197 patches (no multiple of any tile): 32 centroids, int8
        _amm("vit_32_centroids", 12608, 3072, 4, 32, 768),
        # the same images with the table left in fp32
        _amm("vit_fp32_table", 12608, 768, 4, 16, 3072, lut="f32"),
        # the accuracy end of the reference's centroid sweep
        _amm("amm_64_centroids", 8192, 768, 4, 64, 3072),
        # one scale per codebook, the finer quantisation of the benchmark configuration
        _amm("per_codebook_scale", 8192, 3072, 4, 16, 768, scale_group=1),
        # a program that keeps its activations in ordinary host memory
        {"name": "host_buffers", "kind": "host", "n": 8192, "k": 768, "v": 4, "c": 16, "m": 3072},
        # BERT-base, 12 layers, 32 sentences of 128 tokens, launched op by op
        {"name": "bert_base_forward", "kind": "forward", "batch": 32, "seq": 128, "heads": 12, "ffn": 3072, "layers": 12,
         "v": 4, "c": 16, "graph": False},
        # one BERT-large layer, 64 sentences of 128 tokens, replayed from a graph as a server does
        {"name": "bert_large_layer", "kind": "forward", "batch": 64, "seq": 128, "heads": 16, "ffn": 4096, "layers": 1,
         "v": 4, "c": 16, "graph": True},
        # converting one feed-forward matrix of BERT-base
        {"name": "lutgen", "kind": "lutgen", "k": 768, "v": 4, "c": 16, "m": 3072},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


# gathered entries and activation bytes of the largest listed operator, which no drawn one exceeds
_MOST_ENTRIES = 32768 * 256 * 4096
_MOST_BYTES = 4 * 32768 * (1024 + 4096)


def _draw_amm(rng):
    v = rng.choice([2, 4, 4, 4, 8, 16, 32])
    c = rng.choice([8, 16, 16, 16, 16, 24, 32, 64, 128])
    if rng.random() < 0.6:   # model shapes: hidden to hidden, to the feed-forward width and back
        hidden = rng.choice([768, 1024, 1280, 2048])
        k, m = rng.choice([(hidden, hidden), (hidden, 3 * hidden), (hidden, 4 * hidden), (4 * hidden, hidden)])
    else:                    # anything, odd widths among them
        k, m = v * _log(rng, 24, min(1000, 8192 // v)), _log(rng, 64, 4096)
    lut, group = rng.choice([("i8", 0), ("i8", 0), ("i8", 0), ("f32", 0), ("i8", 1)])
    if lut == "f32" or group:
        c = min(c, 32)
    dearer = 8 if c > 32 or lut == "f32" or group else 2 if c > 16 else 1   # an entry's cost beside the 16-centroid int8 one's
    n = min(_log(rng, 1, 32768), _MOST_ENTRIES // (dearer * (k // v) * m), _MOST_BYTES // (4 * (k + m)))
    if rng.random() < 0.4 and n >= 256:
        n = n // 128 * 128
    return {"kind": "amm", "n": n, "k": k, "v": v, "c": c, "m": m, "lut": lut, "scale_group": group, "chain": False}


def draw(rng):
    kind = rng.choice(["amm"] * 7 + ["host", "forward", "forward", "lutgen"])
    if kind == "amm":
        return _draw_amm(rng)
    if kind == "host":
        k, m = rng.choice([(768, 768), (768, 3072), (3072, 768), (1024, 4096)])
        return {"kind": "host", "n": _log(rng, 16, 8192), "k": k, "v": rng.choice([2, 4, 8]), "c": rng.choice([8, 16, 32]), "m": m}
    if kind == "forward":
        heads, ffn = rng.choice([(12, 3072), (16, 4096)])
        seq = rng.choice([17, 64, 128, 197, 264, 512])
        layers = rng.choice([1, 2, 4])
        batch = _log(rng, 1, max(1, 8192 // (seq * layers)))
        return {"kind": "forward", "batch": batch, "seq": seq, "heads": heads, "ffn": ffn, "layers": layers,
                "v": rng.choice([2, 4, 4, 8]), "c": rng.choice([8, 16, 16]), "graph": rng.random() < 0.5}
    k, m = rng.choice([(768, 768), (768, 3072), (3072, 768), (1024, 4096), (768, 1001)])
    return {"kind": "lutgen", "k": k, "v": rng.choice([2, 4, 8, 16]), "c": rng.choice([8, 16, 32, 64]), "m": m}


def _table(rng, k, v, c, m, lut, scale_group):
    """centroids, table, scales of one operator (the table on the CPU, in numpy)."""
    cent = rng.standard_normal((k // v, c, v), dtype=np.float32)
    weight = rng.standard_normal((k, m), dtype=np.float32) * np.float32(0.02)
    full = np.matmul(cent, weight.reshape(k // v, v, m))
    if lut == "f32":
        return cent, full, None
    if scale_group:
        scales = np.abs(full).max(axis=(1, 2)) / np.float32(127)
        each = scales[:, None, None]
    else:
        scales = each = np.float32(np.abs(full).max() / np.float32(127))
    return cent, np.clip(np.rint(full / each), -128, 127).astype(np.int8), scales


def _features(seed, n, k):
    return torch.randn((n, k), device="cuda", generator=torch.Generator(device="cuda").manual_seed(seed))


def prepare(case, seed):
    ctx, rng, kind = _ctx(), np.random.default_rng(seed), case["kind"]
    state = {"kind": kind, "ctx": ctx}
    if kind == "amm":
        shapes = [(case["k"], case["m"])] + ([(case["m"], case["k"])] if case["chain"] else [])
        state["ops"] = []
        for i, (k, m) in enumerate(shapes):
            cent, table, scales = _table(rng, k, case["v"], case["c"], m, case["lut"], case["scale_group"])
            bias = rng.standard_normal(m, dtype=np.float32)
            op = ctx.amm(cent, table, scales, bias, max_n=case["n"], scale_group=case["scale_group"])
            state["ops"].append((op, _features(seed + 1000 * i, case["n"], k), torch.empty((case["n"], m), device="cuda")))
    elif kind == "host":
        cent, table, scales = _table(rng, case["k"], case["v"], case["c"], case["m"], "i8", 0)
        bias = rng.standard_normal(case["m"], dtype=np.float32)
        state["op"] = ctx.amm(cent, table, scales, bias, max_n=case["n"])
        state["x"] = rng.standard_normal((case["n"], case["k"]), dtype=np.float32)
        state["out"] = np.zeros((case["n"], case["m"]), np.float32)
    elif kind == "forward":
        from pim_dl_asplos_amd import transformer
        d, f, v, c = 64 * case["heads"], case["ffn"], case["v"], case["c"]
        p = transformer.TransformerParams(case["seq"], case["batch"], case["heads"], 64, d, f, case["layers"])
        for op, (k, m) in {"q": (d, d), "k": (d, d), "v": (d, d), "o": (d, d), "ffn1": (d, f), "ffn2": (f, d)}.items():
            p.shapes[op] = transformer.AmmShape(k // v, c, k, m)
        state["model"] = transformer.Transformer(ctx, _package, transformer.synth_layers(p, ctx, _package, seed=seed), p)
        state["x"] = _features(seed, p.n, d)
        if case["graph"]:
            state["graph"], state["into"], state["from"] = state["model"].capture(state["x"])
    else:
        state["cent"] = rng.standard_normal((case["k"] // case["v"], case["c"], case["v"]), dtype=np.float32)
        state["weight"] = rng.standard_normal((case["k"], case["m"]), dtype=np.float32) * np.float32(0.02)
    return state


def run(state):
    kind = state["kind"]
    if kind == "amm":
        for op, x, out in state["ops"]:
            op.run_ptr(x.data_ptr(), x.shape[0], out.data_ptr())
        return [out for _, _, out in state["ops"]]
    if kind == "host":
        return state["op"].run(state["x"], state["out"])
    if kind == "forward":
        if "graph" in state:
            state["into"].copy_(state["x"])
            state["graph"].replay()
            return state["from"]
        return state["model"].forward(state["x"])
    table, scales = state["ctx"].lutgen(state["cent"], state["weight"])
    return {"table": table, "scales": scales}


def _amm_work(n, k, v, c, m, entry):
    """x, centroids, the table rows that so many tokens can select, and bias read once, the output written once; a
    multiply-add per score and dimension, an add per gathered entry."""
    cb = k // v
    return 4 * n * k + 4 * c * k + entry * cb * min(c, n) * m + 4 * m + 4 * n * m, 2 * n * k * c + n * cb * m


def work(case):
    kind = case["kind"]
    if kind == "lutgen":
        k, v, c, m = case["k"], case["v"], case["c"], case["m"]
        return {"bytes": 4 * k * m + 4 * c * k + (k // v) * c * m, "flops": 2 * c * k * m}
    if kind in ("amm", "host"):
        entry = 4 if case.get("lut") == "f32" else 1
        b, f = _amm_work(case["n"], case["k"], case["v"], case["c"], case["m"], entry)
        if case.get("chain"):
            b2, f2 = _amm_work(case["n"], case["m"], case["v"], case["c"], case["k"], entry)
            b, f = b + b2, f + f2
        return {"bytes": b, "flops": f}
    n, d, ffn, v, c = case["batch"] * case["seq"], 64 * case["heads"], case["ffn"], case["v"], case["c"]
    table = flops = 0
    for k, m in [(d, d)] * 4 + [(d, ffn), (ffn, d)]:
        table += 4 * c * k + (k // v) * c * m + 4 * m
        flops += _amm_work(n, k, v, c, m, 1)[1]
    flops += 4 * n * case["seq"] * d
    return {"bytes": 8 * n * d + case["layers"] * table, "flops": case["layers"] * flops}


def tolerance(case):
    # fp32 tables: 192 to 1536 entries added in descending instead of ascending codebook order differ by 1.1e-7 to
    # 7.0e-7 (largest 1.2e-6 to 5.3e-6 of the root mean square); either is as far from the sum in float64.
    # Everything else is integer sums with a fixed epilogue, or compares activations with centroids, where another
    # rounding could choose another table row: bits stay.
    if case["kind"] == "amm" and case["lut"] == "f32":
        return {"rel": 2.8e-6, "max": 2.1e-5}
    return "exact"
