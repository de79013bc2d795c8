"""The work a user of this library has it do, as cases that can be timed: dense products at decode and prefill, decode
steps of MoE layers as captured graphs, batched expert products of a prefill, token embedding rows, and loading a matrix
(encode, upload, bit-exact verification).  Sizes are those of the benchmark's 35B-A3B-shaped transformer (model width
2048, 256 experts of 512, vocabulary 248320) and of the tests; draw() spreads them over the ranges the layouts take.

listed() / draw(rng) give cases, prepare(case, seed) what a program holds before the call, run(state) one pass."""
from __future__ import annotations

import math

import torch

from orin_qwen_lossless_amd import decode_step, ops

DEVICE = "cuda"
WEIGHT_SCALE = 0.02
# stored bytes per weight of the layouts on N(0, 0.02) weights (sign|mantissa byte + exponent code)
BYTES_PER_WEIGHT = {"huffman": 1.35, "tiles": 1.41, "nibble": 1.51}

K_MODEL, VOCAB = decode_step.K_MODEL, 248320


def listed() -> list[dict]:
    return [
        # one small projection, one token, launched by itself: the 4-bit code, nothing but latency
        {"name": "dense_small_t1", "kind": "dense", "rows": 512, "k": 2048, "tokens": 1, "engine": "mi355x", "dtype": "bf16"},
        # qkv projection of a 2048-token prefill: exact decode + GEMM
        {"name": "dense_qkv_t2048", "kind": "dense", "rows": 5120, "k": 2048, "tokens": 2048, "engine": "mi355x", "dtype": "bf16"},
        # a tensor in the reference's own 32-lane layout (its tools wrote it), FP32 activations
        {"name": "dense_reflayout_f32_t1", "kind": "dense", "rows": 8192, "k": 2048, "tokens": 1, "engine": "llama", "dtype": "f32"},
        # output projection of one decoded token, and of four (speculative verification, small batches)
        {"name": "head_t1", "kind": "dense", "rows": VOCAB, "k": 2048, "tokens": 1, "engine": "mi355x", "dtype": "bf16"},
        {"name": "head_t4", "kind": "dense", "rows": VOCAB, "k": 2048, "tokens": 4, "engine": "mi355x", "dtype": "bf16"},
        # the layers of a decode step as one graph: a single user, and a small serving batch
        {"name": "step_t1", "kind": "step", "layers": 3, "tokens": 1, "mode": "hybrid"},
        {"name": "step_t16", "kind": "step", "layers": 2, "tokens": 16, "mode": "hybrid"},
        # routed experts of one layer over a prompt: a short ragged one on experts in the 4-bit code, then the
        # benchmark's prompt lengths on the default layout
        {"name": "moe_4bit_t77", "kind": "moe", "experts": 256, "mid": 512, "k": 2048, "topk": 8, "tokens": 77, "mode": "nibble"},
        {"name": "moe_t2048", "kind": "moe", "experts": 256, "mid": 512, "k": 2048, "topk": 8, "tokens": 2048, "mode": "hybrid"},
        {"name": "moe_t8192", "kind": "moe", "experts": 256, "mid": 512, "k": 2048, "topk": 8, "tokens": 8192, "mode": "hybrid"},
        # embedding rows of a 513-token prompt out of the compressed vocabulary matrix
        {"name": "embedding_513", "kind": "embedding", "rows": VOCAB, "k": 2048, "tokens": 513},
        # load time: encode on the host, upload, decode on the device and compare every bit (the encoded exponents have
        # no fixed size: the pass gives the decoded weights in their place)
        {"name": "load_16384", "kind": "load", "rows": 16384, "k": 2048},
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng) -> dict:
    """One more case of the same kinds; no larger than the largest listed ones."""
    kind = rng.choice(("dense", "dense", "dense", "step", "moe", "moe", "moe", "embedding", "load"))
    if kind == "dense":
        k = 512 * rng.randint(1, 8)
        engine = rng.choice(("mi355x", "mi355x", "mi355x", "llama"))
        rows = _log_int(rng, 64, min(VOCAB, (1 << 28) // k))
        rows -= rows % rng.choice((1, 8, 16, 32)) if rows > 64 else 0
        tokens = rng.choice((1, _log_int(rng, 1, 16), _log_int(rng, 1, 2048)))
        if rows * k > 1 << 25:
            tokens = min(tokens, 512)
        return {"kind": kind, "rows": rows, "k": k, "tokens": tokens, "engine": engine, "dtype": "f32" if tokens <= 8 and rng.random() < 0.3 else "bf16"}
    if kind == "step":
        return {"kind": kind, "layers": rng.randint(1, 3), "tokens": rng.randint(1, 16), "mode": rng.choice(("hybrid", "hybrid", "nibble"))}
    if kind == "moe":
        experts, mid = rng.choice(((256, 512), (128, 512), (64, 1024), (48, 512)))
        return {"kind": kind, "experts": experts, "mid": mid, "k": 512 * rng.randint(2, 4), "topk": rng.choice((2, 4, 6, 8)),
                "tokens": _log_int(rng, 1, 8192), "mode": rng.choice(("hybrid", "hybrid", "nibble"))}
    if kind == "embedding":
        return {"kind": kind, "rows": 16 * _log_int(rng, 1024, VOCAB // 16), "k": rng.choice((1024, 2048)), "tokens": _log_int(rng, 1, 2048)}
    return {"kind": kind, "rows": 16 * _log_int(rng, 32, 1024), "k": 512 * rng.randint(1, 4)}


def _generator(seed: int) -> torch.Generator:
    return torch.Generator(device=DEVICE).manual_seed(seed)


def _weights(g: torch.Generator, rows: int, k: int) -> torch.Tensor:
    w = torch.empty((rows, k), dtype=torch.bfloat16, device=DEVICE)
    step = max(1, (1 << 27) // k)
    for r in range(0, rows, step):  # FP32 normals in pieces, rounded once
        n = min(step, rows - r)
        w[r: r + n] = torch.randn((n, k), generator=g, device=DEVICE) * WEIGHT_SCALE
    return w


def _encoded(w: torch.Tensor, engine: str = "mi355x", mode: str = "hybrid", n: int = 1) -> ops.Weight:
    rows, k = w.shape
    fmt, unit_rows, chunk_major, frag, wave64 = ops.choose(rows // n, k, n, engine=engine, mode=mode, expert=n > 1)
    plane, aux, meta = ops.encode(w.cpu(), fmt, unit_rows, chunk_major, frag, wave64)
    return ops.upload(plane, aux, meta, DEVICE)


def _activations(g: torch.Generator, *shape: int) -> torch.Tensor:
    return torch.randn(shape, generator=g, device=DEVICE).to(torch.bfloat16)


def prepare(case: dict, seed: int) -> dict:
    ops.init()
    g = _generator(seed)
    kind = case["kind"]
    if kind == "dense":
        w = _encoded(_weights(g, case["rows"], case["k"]), case["engine"])
        x = _activations(g, case["tokens"], case["k"])
        return {"kind": kind, "w": w, "x": x.float() if case["dtype"] == "f32" else x}
    if kind == "step":
        sets, _, _ = decode_step.make_layer_sets(ops, lambda rows, k: _weights(g, rows, k), case["layers"], False, case["mode"])
        x = _activations(g, case["tokens"], K_MODEL)
        step = decode_step.Bf16nStep(ops, sets, None, case["layers"], case["tokens"])
        h = x.clone()  # the captured step reads its input from this buffer
        graph, out = decode_step.capture(step, h)
        return {"kind": kind, "step": step, "graph": graph, "h": h, "x": x, "out": out}
    if kind == "moe":
        e, mid, k = case["experts"], case["mid"], case["k"]
        st = {"kind": kind, "experts": e, "topk": case["topk"]}
        for name, rows, cols in (("gate", mid, k), ("up", mid, k), ("down", k, mid)):
            st[name] = _encoded(_weights(g, e * rows, cols), mode=case["mode"], n=e)
        st["x"] = _activations(g, case["tokens"], k)
        st["logits"] = torch.randn((case["tokens"], e), generator=g, device=DEVICE)
        return st
    if kind == "embedding":
        w = _encoded(_weights(g, case["rows"], case["k"]), mode="huffman")
        return {"kind": kind, "w": w, "ids": torch.randint(0, case["rows"], (case["tokens"],), generator=g, device=DEVICE)}
    src = _weights(g, case["rows"], case["k"]).cpu()
    return {"kind": kind, "src": src, "layout": ops.choose(case["rows"], case["k"], mode="huffman")}


def run(st: dict):
    kind = st["kind"]
    if kind == "dense":
        x = st["x"]
        return ops.linear(x, st["w"]) if x.dtype == torch.bfloat16 else ops.mmv(x, st["w"])
    if kind == "step":
        st["h"].copy_(st["x"])
        st["graph"].replay()
        return st["out"]
    if kind == "moe":
        wts, ids = ops.router_topk(st["logits"], st["topk"])
        return ops.moe_experts(st["x"], st["gate"], st["up"], st["down"], wts, ids, st["experts"]), wts, ids
    if kind == "embedding":
        return ops.embedding(st["ids"], st["w"])
    fmt, unit_rows, chunk_major, frag, wave64 = st["layout"]
    plane, aux, meta = ops.encode(st["src"], fmt, unit_rows, chunk_major, frag, wave64)
    w = ops.upload(plane, aux, meta, DEVICE)
    return w.plane, ops.dequant(w), ops.roundtrip_equal(w, st["src"])


def _dense_layout(rows: int, k: int, engine: str = "mi355x") -> str:
    return "nibble" if ops.choose(rows, k, engine=engine)[0] == ops.FMT_NIBBLE else "huffman"


def _active(experts: int, pairs: int) -> float:
    """Experts that `pairs` uniform picks are expected to touch."""
    return experts * (1.0 - (1.0 - 1.0 / experts) ** pairs)


def work(case: dict) -> dict:
    """Bytes (weights as stored, inputs and outputs once) and operations one pass cannot do without."""
    kind = case["kind"]
    if kind == "dense":
        rows, k, t = case["rows"], case["k"], case["tokens"]
        elem = 4 if case["dtype"] == "f32" else 2
        return {"bytes": rows * k * BYTES_PER_WEIGHT[_dense_layout(rows, k, case["engine"])] + t * (rows + k) * elem, "flops": 2.0 * rows * k * t}
    experts_layout = "nibble" if case.get("mode") == "nibble" else "tiles"
    if kind == "step":
        d, t = decode_step, case["tokens"]
        dense = sum(r * k * BYTES_PER_WEIGHT["nibble"] for r, k, n in d.SHAPES.values() if n == 1)
        one = 3 * d.N_MID * d.K_MODEL
        moe = (_active(d.E, t * d.TOPK) + 1) * one * BYTES_PER_WEIGHT[experts_layout]
        flops = 2.0 * t * (sum(r * k for r, k, n in d.SHAPES.values() if n == 1) + (d.TOPK + 1) * one)
        return {"bytes": case["layers"] * (dense + moe) + 2 * t * d.K_MODEL * 2, "flops": case["layers"] * flops}
    if kind == "moe":
        one, t = 3 * case["mid"] * case["k"], case["tokens"]
        return {"bytes": _active(case["experts"], t * case["topk"]) * one * BYTES_PER_WEIGHT[experts_layout]
                + t * (2 * case["k"] * 2 + case["experts"] * 4 + case["topk"] * 8), "flops": 2.0 * t * case["topk"] * one}
    if kind == "embedding":
        return {"bytes": case["tokens"] * case["k"] * (BYTES_PER_WEIGHT["huffman"] + 2) + 8 * case["tokens"], "flops": 0}
    n = case["rows"] * case["k"]
    return {"bytes": n * (2 + BYTES_PER_WEIGHT["huffman"] + 2), "flops": 0}


def tolerance(case: dict):
    """Embedding rows and loading are exact.  Products: FP32 sums, rounded to BF16 except with FP32 activations; about
    four times the deviation from an FP64 evaluation (dense 1.7e-3, FP32 activations 7e-8, experts 2.4e-3, a step of two
    layers 2.7e-3).  A step may also pick another eighth expert where the router's logits nearly tie: `max`."""
    kind = case["kind"]
    if kind in ("embedding", "load"):
        return "exact"
    if kind == "dense":
        return {"rel": 1e-6, "max": 1e-5} if case["dtype"] == "f32" else {"rel": 7e-3, "max": 2e-2}
    if kind == "moe":
        return {"rel": 1e-2, "max": 5e-2}
    return {"rel": 1.2e-2, "max": 0.5}
