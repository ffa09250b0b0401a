"""The work whose speed matters to a program that uses this package, as measurable cases.

`listed()` names twelve cases of the ranges that `draw()` samples; a case is a dict of plain values whose "kind" is

  gemv     decode projections (DeviceWeights.gemv): one eager call, or a captured graph over the same projection of several
           layers, as a decode step walks them; 1 to 32 activation rows, every format that the planner and the registry use
  layer    the matmuls of one decoder layer through the layer API: norm + q/k/v, output projection, norm + gated MLP
  prefill  prompt processing (DeviceWeights.gemm_bf16 / gemm_f32)
  moe      one mixture-of-experts step: host routing of the router's logits, grouped dispatch
  kv       one layer's OIL4 KV cache through a generation: prompt appended, then per step one token appended and the context read
  flat     the flat-codebook entry points of kernel.py (kernel::oil{4,8}_gemm, production GEMVs, engine quant_gemm)
  encode   the block quantizer on host weights
  decode   whole-tensor dequantization, or rows of an embedding table

Weights are N(0, 0.02) with 1 % of the blocks scaled x8 (a pool of such blocks goes through the block quantizer and tensors are
drawn from the pool), activations N(0, 1)."""
import math

import numpy as np
import torch

import innova_amd as ia
from innova_amd import kernel, layers, moe

WIRE = 256
POOL = 1024                      # distinct blocks per format that a tensor is drawn from

# what a tensor's blocks are: one format, or a mix as {format: share}.  "planner" is FormatPlanner's answer at its default
# 1.50 bits per weight (the more important half SPARK_Q0, the rest OIL1), "spark_mix" the registry's SPARK_MIX_Q0.
MIXES = {
    "planner": {"SPARK_Q0": 0.5, "OIL1": 0.5},
    "spark_mix": {"OIL8_GRP": 0.01, "OIL4_GRP": 0.02, "OIL2_GRP": 0.52, "OIL1_GRP": 0.45},
}


def listed():
    return [
        # the smallest call: a narrow projection, issued eagerly; an odd number of rows and of blocks per row
        {"name": "gemv_small_eager", "kind": "gemv", "fmt": "OIL4", "rows": 1000, "cols": 1280, "m": 1, "tensors": 1},
        # the headline shape: up / gate projection of one token, eight layers of a captured decode step
        {"name": "gemv_oil4_up_m1", "kind": "gemv", "fmt": "OIL4", "rows": 11008, "cols": 4096, "m": 1, "tensors": 8},
        # down projection of a batch of sixteen sequences
        {"name": "gemv_oil4_down_m16", "kind": "gemv", "fmt": "OIL4", "rows": 4096, "cols": 11008, "m": 16, "tensors": 8},
        # the output head of one token
        {"name": "head_oil4_m1", "kind": "gemv", "fmt": "OIL4", "rows": 131072, "cols": 4096, "m": 1, "tensors": 1},
        # a decoder layer at the planner's 1.50 bits per weight
        {"name": "layer_planner_m1", "kind": "layer", "fmt": "planner", "d": 4096, "f": 11008, "m": 1},
        # a smaller layer with a few sequences in flight, no size a power of two
        {"name": "layer_oil4_ragged_m5", "kind": "layer", "fmt": "OIL4", "d": 2816, "f": 7424, "m": 5},
        # a long prompt, bf16 activations
        {"name": "prefill_oil4_2048", "kind": "prefill", "fmt": "OIL4", "rows": 11008, "cols": 4096, "m": 2048, "x": "bf16"},
        # an odd prompt chunk, FP32 activations, weights that mix formats
        {"name": "prefill_planner_ragged", "kind": "prefill", "fmt": "planner", "rows": 5000, "cols": 2816, "m": 437, "x": "f32"},
        # eight experts, 64 tokens, top-2, uneven loads
        {"name": "moe_8x64_top2", "kind": "moe", "d": 4096, "f": 14336, "experts": 8, "tokens": 64, "topk": 2, "z_loss": False},
        # a 2048-token prompt and eight decode steps of one layer's cache
        {"name": "kv_2048_plus_8", "kind": "kv", "prompt": 2048, "steps": 8, "heads": 32, "dim": 128, "block": 64},
        # OIL4Engine::quant_gemm of one token (the engines' k-ordered sums)
        {"name": "engine_oil4_m1", "kind": "flat", "op": "engine4", "m": 1, "n": 4096, "k": 4096},
        # quantizing one projection of a model
        {"name": "encode_oil4", "kind": "encode", "fmt": "OIL4", "numel": 4096 * 4096},
    ]


def _log(rng, lo, hi):
    """An integer of [lo, hi], spread over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


WEIGHT_FMTS = ["OIL4"] * 5 + ["OIL8"] * 2 + ["planner"] * 3 + ["spark_mix"] * 2 + ["OIL2", "SPARK_Q0", "OIL4_GRP", "OIL8_GRP"]
FLAT_OPS = ["oil8", "oil4", "prod_spark", "prod_oil4", "prod_oil8", "engine8", "engine4", "engine2"]


def draw(rng):
    kind = rng.choice(["gemv"] * 7 + ["layer"] * 3 + ["prefill"] * 3 + ["moe"] * 2 + ["kv"] * 2 + ["flat"] * 3 + ["encode"] + ["decode"])
    fmt = rng.choice(WEIGHT_FMTS)
    if kind == "gemv":
        rows, cols = _log(rng, 256, 32768), WIRE * _log(rng, 2, 56)
        m = rng.choice([1, 1, 1, _log(rng, 2, 32)])
        tensors = rng.choice([1, _log(rng, 2, 12)])
        while tensors > 1 and tensors * rows * cols > 400e6:
            tensors -= 1
        return {"kind": kind, "fmt": fmt, "rows": rows, "cols": cols, "m": m, "tensors": tensors}
    if kind == "layer":
        d = WIRE * _log(rng, 3, 16)
        return {"kind": kind, "fmt": fmt, "d": d, "f": WIRE * max(2, int(d / WIRE * rng.uniform(2.0, 3.6))), "m": rng.choice([1, 1, _log(rng, 2, 16)])}
    if kind == "prefill":
        return {"kind": kind, "fmt": fmt, "rows": _log(rng, 500, 11008), "cols": WIRE * _log(rng, 4, 43), "m": _log(rng, 33, 1024), "x": rng.choice(["bf16", "f32"])}
    if kind == "moe":
        d = WIRE * _log(rng, 4, 16)
        return {"kind": kind, "d": d, "f": WIRE * max(2, int(d / WIRE * rng.uniform(1.0, 3.5))), "experts": rng.choice([4, 6, 8]),
                "tokens": _log(rng, 1, 64), "topk": rng.choice([1, 2]), "z_loss": rng.random() < 0.3}
    if kind == "kv":
        return {"kind": kind, "prompt": _log(rng, 1, 2048), "steps": rng.randint(0, 8), "heads": rng.choice([4, 5, 8, 16, 32]),
                "dim": rng.choice([64, 80, 128]), "block": rng.choice([32, 64, 64, 128])}
    if kind == "flat":
        return {"kind": kind, "op": rng.choice(FLAT_OPS), "m": rng.choice([1, 1, _log(rng, 2, 8)]), "n": _log(rng, 256, 11008), "k": 4 * _log(rng, 128, 1536)}
    if kind == "encode":
        return {"kind": kind, "fmt": fmt, "numel": _log(rng, 100_000, 12_000_000)}
    rows, cols = _log(rng, 256, 16384), WIRE * _log(rng, 2, 32)
    return {"kind": kind, "fmt": fmt, "rows": rows, "cols": cols, "ids": rng.choice([0, _log(rng, 1, 512)])}


# ---- inputs

def _weights(rng, n):
    w = rng.standard_normal(n, dtype=np.float32) * np.float32(0.02)
    full = w[: n // WIRE * WIRE].reshape(-1, WIRE)
    full[rng.random(len(full)) < 0.01] *= np.float32(8.0)
    return w


def _formats(rng, fmt, nblocks):
    """One format id per block, in the mix's shares."""
    if fmt not in MIXES:
        return np.full(nblocks, int(ia.Format[fmt]), np.uint8)
    ids = [int(ia.Format[f]) for f in MIXES[fmt]]
    return np.array(ids, np.uint8)[np.searchsorted(np.cumsum(list(MIXES[fmt].values()))[:-1], rng.random(nblocks))]


class _Pool:
    """POOL quantized blocks per format of `fmt`, and tensors drawn from them."""

    def __init__(self, rng, fmt):
        self.rng, self.fmt = rng, fmt
        self.names = list(MIXES.get(fmt, {fmt: 1.0}))
        self.blocks = {}
        for name in self.names:
            payload, blocks = ia.block_codec.quantize_tensor(_weights(rng, POOL * WIRE), ia.Format[name])
            self.blocks[int(ia.Format[name])] = (payload.reshape(POOL, -1), blocks[0])

    def tensor(self, rows, cols):
        n = rows * cols // WIRE
        fm = _formats(self.rng, self.fmt, n)
        desc = np.zeros(n, ia._lib.BLOCK_DTYPE)
        desc["nw"], desc["fmt"] = WIRE, fm
        parts, at = [], 0
        for f, (pool, first) in self.blocks.items():
            where = np.flatnonzero(fm == f)
            size = pool.shape[1]
            parts.append(pool[self.rng.integers(0, POOL, where.size)].reshape(-1))
            desc["cb_bytes"][where], desc["idx_bytes"][where] = first["cb_bytes"], first["idx_bytes"]
            desc["cb_off"][where] = at + size * np.arange(where.size, dtype=np.uint64)
            desc["idx_off"][where] = desc["cb_off"][where] + first["cb_bytes"]
            at += size * where.size
        return ia.DeviceWeights.from_blocks(parts[0] if len(parts) == 1 else np.concatenate(parts), desc, rows, cols)


def prepare(case, seed):
    rng = np.random.default_rng(seed)
    gen = torch.Generator(device="cuda").manual_seed(seed)

    def acts(*shape):
        return torch.randn(*shape, generator=gen, device="cuda")

    def codes(*shape):
        return torch.randint(0, 256, shape, generator=gen, device="cuda", dtype=torch.uint8)

    s = dict(case)
    kind = case["kind"]
    if kind == "gemv":
        pool = _Pool(rng, case["fmt"])
        ws = s["w"] = [pool.tensor(case["rows"], case["cols"]) for _ in range(case["tensors"])]
        xs = s["xs"] = [acts(case["m"], case["cols"]) for _ in ws]
        if len(ws) > 1:                                   # a decode step is captured once and replayed per token
            ys = s["ys"] = [torch.empty(case["m"], case["rows"], device="cuda") for _ in ws]
            stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
            stream.wait_stream(torch.cuda.current_stream())
            with torch.cuda.stream(stream):
                ws[0].gemv(xs[0], out=ys[0])
            torch.cuda.synchronize()
            with torch.cuda.graph(graph, stream=stream):
                for w, x, y in zip(ws, xs, ys):
                    w.gemv(x, out=y)
            s["graph"] = graph
    elif kind == "layer":
        pool, d, f, m = _Pool(rng, case["fmt"]), case["d"], case["f"], case["m"]
        s.update(qkv=pool.tensor(3 * d, d), o=pool.tensor(d, d), gate_up=pool.tensor(2 * f, d), down=pool.tensor(d, f),
                 h=acts(m, d), att=acts(m, d), norm1=acts(d) * 0.1, norm2=acts(d) * 0.1)
    elif kind == "prefill":
        s["w"] = _Pool(rng, case["fmt"]).tensor(case["rows"], case["cols"])
        s["act"] = acts(case["m"], case["cols"]).to(torch.bfloat16 if case["x"] == "bf16" else torch.float32)
    elif kind == "moe":
        pool, d, f = _Pool(rng, "OIL4"), case["d"], case["f"]
        s["w"] = [moe.ExpertFFN(pool.tensor(f, d), pool.tensor(f, d), pool.tensor(d, f)) for _ in range(case["experts"])]
        s["act"] = acts(case["tokens"], d)
        logits = rng.standard_normal((case["tokens"], case["experts"])).astype(np.float32)
        logits[:, 0] += 1.0                               # uneven loads
        s["logits"] = logits
        s["ws"] = None if case["z_loss"] else moe.moe_workspace(s["act"], s["w"], case["topk"])
    elif kind == "kv":
        p, n, h, d = case["prompt"], case["steps"], case["heads"], case["dim"]
        s["cache"] = ia.OIL4KVCache(1, p + n, h, d, case["block"])
        s["k"], s["v"] = acts(1, h, p, d), acts(1, h, p, d)
        s["step_k"], s["step_v"] = [acts(1, h, 1, d) for _ in range(n)], [acts(1, h, 1, d) for _ in range(n)]
    elif kind == "flat":
        m, n, k, op = case["m"], case["n"], case["k"], case["op"]
        bits = {"oil8": 8, "prod_oil8": 8, "engine8": 8, "prod_spark": 2, "engine2": 2}.get(op, 4)
        pairs = m * n if op == "oil4" else n              # kernel::oil4_gemm holds one packed row per (m, n) pair
        s["codes"] = codes((pairs * k * bits + 7) // 8)
        s["act"] = acts(n if op == "oil4" else m, k)
        levels = torch.sort(acts(1 << (bits if op != "prod_spark" else 4))).values
        s["cb"] = levels.to(torch.float16).view(torch.int16) if op in ("oil4", "prod_oil4") else levels
    elif kind == "encode":
        s["weights"] = _weights(rng, case["numel"])
        s["formats"] = _formats(rng, case["fmt"], -(-case["numel"] // WIRE))
    else:
        s["w"] = _Pool(rng, case["fmt"]).tensor(case["rows"], case["cols"])
        if case["ids"]:
            s["rows_wanted"] = torch.randint(0, case["rows"], (case["ids"],), generator=gen, device="cuda", dtype=torch.int32)
    return s


# ---- one pass

def run(s):
    kind = s["kind"]
    if kind == "gemv":
        if "graph" in s:
            s["graph"].replay()
            return s["ys"]
        return s["w"][0].gemv(s["xs"][0])
    if kind == "layer":
        qkv = layers.gemv_rmsnorm(s["qkv"], s["h"], s["norm1"])
        o = s["o"].gemv(s["att"])                         # attention itself is not part of this package
        return qkv, o, layers.mlp_step(s["gate_up"], s["down"], o, norm_w=s["norm2"])
    if kind == "prefill":
        return s["w"].gemm_bf16(s["act"]) if s["x"] == "bf16" else s["w"].gemm_f32(s["act"])
    if kind == "moe":
        _, idx, wgt = moe.softmax_with_topk(s["logits"], s["topk"])
        return moe.moe_dispatch_batched(s["act"], s["w"], idx, wgt, want_z_loss=s["z_loss"], workspace=s["ws"])
    if kind == "kv":
        cache, n = s["cache"], s["prompt"]
        cache.clear()
        cache.append(0, s["k"], s["v"])
        out = None
        for k, v in zip(s["step_k"], s["step_v"]):
            cache.append(0, k, v)
            n += 1
            out = cache.get_range(0, 0, n)
        return out if out is not None else cache.get_range(0, 0, n)
    if kind == "flat":
        m, n, k, op = s["m"], s["n"], s["k"], s["op"]
        if op == "oil8":
            return kernel.oil8_gemm(s["codes"], s["cb"], s["act"], m, n, k)
        if op == "oil4":
            return kernel.oil4_gemm(s["codes"], s["cb"], s["act"], m, n, k)
        if op == "prod_spark":                            # the production forms count weight rows first, then activation rows
            return kernel.gemv_spark_batch(s["codes"], 0.02, s["act"], n, m, k)
        if op == "prod_oil4":
            return kernel.gemv_oil4_batch(s["codes"], s["cb"], 0.02, s["act"], n, m, k)
        if op == "prod_oil8":
            return kernel.gemv_oil8_batch(s["codes"], s["cb"], 0.02, s["act"], n, m, k)
        return kernel.engine_quant_gemm(int(op[6:]), s["act"], s["codes"], s["cb"], m, n, k)
    if kind == "encode":
        payload, blocks = ia.block_codec.quantize_tensor(s["weights"], s["formats"])
        return payload, blocks["cb_off"], blocks["idx_off"], blocks["idx_bytes"]
    return layers.embed_rows(s["w"], s["rows_wanted"]) if s["ids"] else s["w"].dequant()


# ---- what a pass cannot do without

def _payload(fmt, numel):
    """Bytes of `numel` weights in that format or mix (share-weighted full-block sizes)."""
    return numel / WIRE * sum(share * ia.FULL_BLOCK_BYTES[ia.Format[f]] for f, share in MIXES.get(fmt, {fmt: 1.0}).items())


def work(case):
    kind = case["kind"]
    m = case.get("m", 1)
    if kind in ("gemv", "prefill"):
        n, k, t = case["rows"], case["cols"], case.get("tensors", 1)
        x_bytes = 2 if case.get("x") == "bf16" else 4
        return {"bytes": t * (_payload(case["fmt"], n * k) + m * (x_bytes * k + 4 * n)), "flops": 2.0 * t * m * n * k}
    if kind == "layer":
        d, f = case["d"], case["f"]
        numel = 3 * d * d + d * d + 2 * f * d + d * f
        return {"bytes": _payload(case["fmt"], numel) + 4 * (m * (d + 3 * d + d + d + d) + 2 * d), "flops": 2.0 * m * numel}
    if kind == "moe":
        d, f, e, pairs = case["d"], case["f"], case["experts"], case["tokens"] * case["topk"]
        used = e * (1.0 - (1.0 - 1.0 / e) ** pairs)       # experts that some token is expected to visit
        return {"bytes": used * _payload("OIL4", 3 * d * f) + 8 * case["tokens"] * d, "flops": 2.0 * pairs * 3 * d * f}
    if kind == "kv":
        p, n, token = case["prompt"], case["steps"], 2 * case["heads"] * case["dim"]
        stored = 0.5 + 32.0 / case["block"]               # bytes per value: its code, and its share of sixteen FP16 centroids
        reads = sum(p + i + 1 for i in range(n)) if n else p
        return {"bytes": (p + n) * token * (4 + stored) + reads * token * (4 + stored), "flops": (p + n) * token * 48.0}
    if kind == "flat":
        n, k, op = case["n"], case["k"], case["op"]
        bits = {"oil8": 8, "prod_oil8": 8, "engine8": 8, "prod_spark": 2, "engine2": 2}.get(op, 4)
        rows, pairs = (n, m * n) if op == "oil4" else (m, n)
        return {"bytes": pairs * k * bits / 8 + 4 * (rows * k + m * n), "flops": 2.0 * m * n * k}
    if kind == "encode":
        return {"bytes": 4 * case["numel"] + _payload(case["fmt"], case["numel"]), "flops": 4.0 * case["numel"]}
    numel = (case["ids"] or case["rows"]) * case["cols"]
    return {"bytes": 4 * numel + _payload(case["fmt"], numel), "flops": 1.0 * numel}


def tolerance(case):
    kind = case["kind"]
    if kind in ("kv", "encode", "decode") or (kind == "flat" and case["op"].startswith("engine")):
        return "exact"                                    # bytes, or values that the reference's own order of operations fixes
    if kind == "prefill":
        return {"rel": 2e-3, "max": 2e-2}                 # bf16 operands: one rounding per weight and activation
    return {"rel": 1e-5}                                  # FP32 sums
