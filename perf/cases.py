"""Workloads of the tiered decode path that its speed is measured on.

Every case is work that a user of this package has it do, through the C ABI or
the Python API: decode attention at the benchmark's model shapes (captured in a
HIP graph, as a serving loop replays it, or called from Python), batched ragged
decode, engine decode steps, a prompt's prefill with its first decode step, and
the bulk quantisers and dequantisers. Inputs are synthetic and made on the GPU
from a seed: N(0, 1) values with four key channels per KV head scaled by 8, the
key outliers that 2-bit caches meet. Packed tiers are built here in torch, so a
case's inputs do not depend on the quantisers being measured.
"""
import ctypes
import math
import random

import torch

from tritiercache_amd import _C, _lib
from tritiercache_amd.cache import TriTierCache

SINK = 4  # sink tokens of every engine (the package's constant)
RECENT = 256  # recent window of the HF patch and the benchmark
HEAVY = 0.05  # heavy-hitter share of the HF patch and the benchmark
DEFER_MIN_LAYERS = 16  # models of at least this many layers defer the mean weights, as the benchmark does


# ---------------------------------------------------------------------------
# Cases
# ---------------------------------------------------------------------------
def _tiers(ctx):
    """FP32 tokens, packed blocks of 16 and masked slots of a context: sinks, recent window and heavy hitters in
    FP32, the rest packed, the last block filled up with masked slots."""
    dense = SINK + RECENT + math.ceil(HEAVY * ctx)
    packed = max(ctx - dense, 0)
    blocks = (packed + 15) // 16
    return dense, blocks, blocks * 16 - packed


def _attention(hq, hkv, d, ctx, layers, meta, kgs=16, call="graph", weights=True):
    dense, blocks, masked = _tiers(ctx)
    if kgs == 32:
        masked += 16 * (blocks % 2)
        blocks = (blocks + 1) // 2
    return {"kind": "attention", "hq": hq, "hkv": hkv, "d": d, "dense": dense, "blocks": blocks, "masked": masked,
            "kgs": kgs, "meta": meta, "layers": layers, "call": call, "weights": weights}


def listed():
    return [
        # The reference's published call: 32/8 heads, 260 FP32 tokens and 20 packed blocks, one call from Python.
        # What a short chat context costs: launches and the host path.
        {"name": "fused-580", "kind": "attention", "hq": 32, "hkv": 8, "d": 128, "dense": 260, "blocks": 20,
         "masked": 0, "kgs": 16, "meta": "fp32", "layers": 1, "call": "python", "weights": True},
        # The headline benchmark: a Llama-3-8B decode step over 32 layers at 32k context.
        {"name": "llama3-8b-32k", **_attention(32, 8, 128, 32768, 32, "fp32")},
        # Multi-head attention (one query head per KV head) at 8k, FP16 metadata.
        {"name": "mha-8k", **_attention(32, 32, 128, 8192, 8, "fp16")},
        # head_dim 64 (the TinyLlama / SmolLM head size) at 32k, blocks of 32 tokens.
        {"name": "hd64-32k", **_attention(32, 8, 64, 32768, 16, "fp16", kgs=32)},
        # head_dim 256 with two query heads per KV head (the Gemma-2-9B shape) at 8k.
        {"name": "gemma2-hd256-8k", **_attention(16, 8, 256, 8192, 16, "fp32")},
        # head_dim 80 with 32/32 heads (the Phi-2 shape) at 2k.
        {"name": "phi2-hd80-2k", **_attention(32, 32, 80, 2048, 32, "fp32")},
        # Serving: one layer's decode step of 16 ragged sequences (Mistral-7B heads), called from Python.
        {"name": "mistral-batch16", "kind": "batched", "hq": 32, "hkv": 8, "d": 128, "seqs": 16, "shortest": 2048,
         "longest": 32768, "lengths": 7, "kgs": 16, "meta": "fp32"},
        # A decode step of four layers through the engine with 4k prompts, TriTierCache.step per layer (the class's
        # defaults: FP16 metadata, blocks of 16).
        {"name": "engine-4k", "kind": "engine", "hq": 32, "hkv": 8, "d": 128, "prompt": 4096, "layers": 4, "kgs": 16,
         "meta": "fp16", "deferred": False},
        # Long-context decode: four layers of the Qwen2-7B heads with 128k prompts, each layer's score feedback in
        # the next layer's launch, as the HF patch chains its layers.
        {"name": "engine-128k", "kind": "engine", "hq": 28, "hkv": 4, "d": 128, "prompt": 131072, "layers": 4,
         "kgs": 16, "meta": "fp32", "deferred": True},
        # A new prompt of one layer: a fresh cache, the bulk ingest of 16k tokens and the first decode step.
        {"name": "prefill-16k", "kind": "prefill", "hq": 32, "hkv": 8, "d": 128, "prompt": 16384, "kgs": 16,
         "meta": "fp16"},
        # Packing the keys and values of a 32k context (encode), FP16 metadata.
        {"name": "quantize-32k", "kind": "quantize", "h": 8, "d": 128, "blocks": 2048, "kgs": 16, "meta": "fp16"},
        # Unpacking a 16k context of 32 heads (decode), FP32 metadata and blocks of 32 tokens.
        {"name": "dequantize-16k", "kind": "dequantize", "h": 32, "d": 128, "blocks": 512, "kgs": 32, "meta": "fp32"},
    ]


# (query heads, KV heads, head_dim) of the repository's benchmark configurations and tests
_HEADS = ((32, 8, 128), (32, 32, 128), (28, 4, 128), (40, 10, 128), (16, 8, 128), (32, 8, 64), (14, 2, 64),
          (9, 3, 64), (16, 8, 256), (8, 4, 256), (32, 32, 80), (32, 32, 96), (12, 4, 96))


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("attention", "attention", "attention", "batched", "engine", "prefill", "quantize",
                       "dequantize"))
    kgs, meta = rng.choice((16, 16, 32)), rng.choice(("fp32", "fp16"))
    if kind == "attention":
        hq, hkv, d = rng.choice(_HEADS)
        if rng.random() < 0.3:
            c = _attention(hq, hkv, d, _log_int(rng, 300, 16384), 1, meta, kgs, "python", rng.random() < 0.7)
        else:
            c = _attention(hq, hkv, d, _log_int(rng, 700, 32768), 1, meta, kgs, "graph", rng.random() < 0.8)
            c["layers"] = max(2, min(32, int(4e8 / work(c)["bytes"])))
        return c
    if kind == "batched":
        hq, hkv, d = rng.choice(((32, 8, 128), (28, 4, 128), (16, 8, 128), (32, 32, 128)))
        seqs = rng.randint(2, 24)
        longest = _log_int(rng, 1024, 20000 if hkv <= 8 else 5000)
        return {"kind": "batched", "hq": hq, "hkv": hkv, "d": d, "seqs": seqs, "shortest": max(300, longest // 12),
                "longest": longest, "lengths": rng.randint(1, 1 << 20), "kgs": kgs, "meta": meta}
    if kind == "engine":
        hq, hkv, d = rng.choice(_HEADS)
        return {"kind": "engine", "hq": hq, "hkv": hkv, "d": d, "prompt": _log_int(rng, 400, 65536 if hkv <= 8 else 12000),
                "layers": rng.randint(1, 4), "kgs": kgs, "meta": meta, "deferred": rng.random() < 0.5}
    if kind == "prefill":
        hq, hkv, d = rng.choice(_HEADS)
        return {"kind": "prefill", "hq": hq, "hkv": hkv, "d": d, "prompt": _log_int(rng, 300, 32768 if hkv <= 8 else 8192),
                "kgs": kgs, "meta": meta}
    h, d = rng.choice(((8, 128), (4, 128), (32, 128), (10, 128), (8, 64), (3, 64), (8, 256), (32, 80), (32, 96)))
    blocks = _log_int(rng, 1, (1 << 26) // (h * d * 2 * kgs))
    return {"kind": kind, "h": h, "d": d, "blocks": blocks, "kgs": kgs, "meta": meta}


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------
def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _keys(g, n, h, d):
    k = torch.randn((n, h, d), generator=g, device="cuda")
    for j in range(h):
        k[:, j, torch.randperm(d, generator=g, device="cuda")[:4]] *= 8.0
    return k


def _values(g, n, h, d):
    return torch.randn((n, h, d), generator=g, device="cuda")


def _scales(lo, hi, meta):
    """(scale in FP32, stored scale, stored zero) of 2-bit groups with these extremes."""
    # a tensor of threes: torch turns a division by a number into a product with its rounded reciprocal
    s = ((hi - lo) / torch.full_like(hi, 3.0)).clamp_min(1e-9)
    if meta == "fp16":
        return s, s.to(torch.float16).view(torch.uint16), lo.to(torch.float16).view(torch.uint16)
    return s, s, lo


def _words(codes, dim):
    """16 codes along `dim` to one int32 each, code i at bits 2 i."""
    shift = (2 * torch.arange(16, device=codes.device, dtype=torch.int32)).view([16 if i == dim else 1
                                                                                for i in range(codes.dim())])
    return (codes.to(torch.int32) << shift).sum(dim, dtype=torch.int32)


def _pack_keys(k, kgs, meta):
    """Keys [blocks * kgs, H, D], per channel of a block: words [blocks, kgs / 16, H, D], scale and zero [blocks, H, D]."""
    _, h, d = k.shape
    x = k.view(-1, kgs, h, d)
    lo = x.amin(1)
    s, scale, zero = _scales(lo, x.amax(1), meta)
    codes = torch.round((x - lo[:, None]) / s[:, None]).clamp_(0, 3)
    return _words(codes.view(-1, kgs // 16, 16, h, d), 2), scale, zero


def _pack_values(v, meta):
    """Values [tokens, H, D], per token and head: words [tokens, H, D / 16], scale and zero [tokens, H]."""
    n, h, d = v.shape
    lo = v.amin(2)
    s, scale, zero = _scales(lo, v.amax(2), meta)
    codes = torch.round((v - lo[..., None]) / s[..., None]).clamp_(0, 3)
    return _words(codes.view(n, h, d // 16, 16), 3), scale, zero


def _pbs(g, case, blocks):
    h, d, kgs = case["hkv"], case["d"], case["kgs"]
    n = blocks * kgs
    kp, ks, kz = _pack_keys(_keys(g, n, h, d), kgs, case["meta"])
    vp, vs, vz = _pack_values(_values(g, n, h, d), case["meta"])
    return {"kp": kp, "ks": ks, "kz": kz, "vp": vp, "vs": vs, "vz": vz}


def _sequence(g, case, dense, blocks, masked):
    """One layer's (or sequence's) tier tables and query."""
    h, d = case["hkv"], case["d"]
    t = {"q": torch.randn((case["hq"], d), generator=g, device="cuda"), "dk": _keys(g, dense, h, d),
         "dv": _values(g, dense, h, d), **_pbs(g, case, blocks)}
    t["ids"] = torch.arange(dense, dense + blocks * case["kgs"], dtype=torch.int64, device="cuda")
    if masked:
        t["ids"][-masked:] = -1
    return t


# ---------------------------------------------------------------------------
# Decode attention
# ---------------------------------------------------------------------------
def _stream():
    return ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)


_TIERS = ("q", "dk", "dv", "kp", "ks", "kz", "vp", "vs", "vz", "ids")


def _prepare_attention(case, seed):
    g = _generator(seed)
    n, hq, d = case["dense"] + case["blocks"] * case["kgs"], case["hq"], case["d"]
    s = {"case": case, "layers": [_sequence(g, case, case["dense"], case["blocks"], case["masked"])
                                  for _ in range(case["layers"])]}
    s["out"] = torch.zeros((case["layers"], hq, d), device="cuda")
    s["mean"] = torch.zeros((case["layers"], n), device="cuda") if case["weights"] else None
    if case["call"] == "graph":
        _capture(s)
    return s


def _capture(s):
    """The step over all layers as a HIP graph, through the C ABI with workspaces of the caller."""
    case, lib = s["case"], _lib.load()
    hq, hkv, d, kgs, nd, nb = (case[k] for k in ("hq", "hkv", "d", "kgs", "dense", "blocks"))
    fp16, mean = int(case["meta"] == "fp16"), case["weights"]
    size = lib.tt_fused_attention_workspace_bytes(nd, nb, hq, hkv, d, kgs, int(mean))
    deferred = mean and case["layers"] >= DEFER_MIN_LAYERS
    s["ws"] = ws = [torch.empty(size, dtype=torch.uint8, device="cuda") for _ in range(2 if deferred else 1)]

    def tiers(t):
        p = [t[k].data_ptr() for k in _TIERS]
        return [*p[:3], nd, *p[3:], nb, hq, hkv, d]

    def per_layer(i):
        rc = lib.tt_fused_attention_decode_ws(*tiers(s["layers"][i]), s["out"][i].data_ptr(),
                                              s["mean"][i].data_ptr() if mean else None, kgs, fp16, ws[0].data_ptr(),
                                              size, _stream())
        _lib.check(rc, "decode")

    def step():
        if not deferred:
            for i in range(case["layers"]):
                per_layer(i)
            return
        for i, t in enumerate(s["layers"]):
            w, p = ws[i % 2].data_ptr(), ws[(i + 1) % 2].data_ptr()
            q, out = t["q"].data_ptr(), s["out"][i].data_ptr()
            _lib.check(lib.tt_attention_partials(*tiers(t), kgs, fp16, 1, w, size, _stream()), "partials")
            if i == 0:
                rc = lib.tt_attention_finalize(q, nd, nb, hq, hkv, d, out, None, kgs, fp16, 1, w, size, _stream())
            else:
                rc = lib.tt_attention_finalize_deferred(q, nd, nb, hq, hkv, d, out, kgs, fp16, w, size, nd, nb,
                                                        s["mean"][i - 1].data_ptr(), p, size, _stream())
            _lib.check(rc, "finalize")
        rc = lib.tt_attention_finalize(q, nd, nb, hq, hkv, d, None, s["mean"][-1].data_ptr(), kgs, fp16, 1, w, size,
                                       _stream())
        _lib.check(rc, "mean weights")

    step()  # loads the kernels before the capture
    torch.cuda.synchronize()
    s["graph"] = torch.cuda.CUDAGraph()
    with torch.cuda.graph(s["graph"]):
        step()
    s["out"].zero_()
    if mean:
        s["mean"].zero_()


def _run_attention(s):
    if "graph" in s:
        s["graph"].replay()
    else:
        case = s["case"]
        for i, t in enumerate(s["layers"]):
            _C.fused_attention_decode(t["q"], t["dk"], t["dv"], case["dense"], t["kp"], t["ks"], t["kz"], t["vp"],
                                      t["vs"], t["vz"], t["ids"], case["blocks"], case["hq"], case["hkv"], case["d"],
                                      s["out"][i], s["mean"][i] if case["weights"] else None, case["kgs"], case["meta"])
    return [s["out"], s["mean"]] if s["case"]["weights"] else [s["out"]]


# ---------------------------------------------------------------------------
# Batched ragged decode
# ---------------------------------------------------------------------------
def _lengths(case):
    r = random.Random(case["lengths"])
    return [_tiers(r.randint(case["shortest"], case["longest"])) for _ in range(case["seqs"])]


def _blocks_of(case, tiers):
    dense, blocks, masked = tiers
    if case["kgs"] == 32:
        return dense, (blocks + 1) // 2, masked + 16 * (blocks % 2)
    return dense, blocks, masked


def _prepare_batched(case, seed):
    g = _generator(seed)
    batch = []
    for tiers in _lengths(case):
        dense, blocks, masked = _blocks_of(case, tiers)
        t = _sequence(g, case, dense, blocks, masked)
        batch.append({"Q": t["q"], "dense_K": t["dk"], "dense_V": t["dv"], "dense_count": dense,
                      "PBS_K_Packed": t["kp"], "PBS_K_Scales": t["ks"], "PBS_K_Zeroes": t["kz"],
                      "PBS_V_Packed": t["vp"], "PBS_V_Scales": t["vs"], "PBS_V_Zeroes": t["vz"],
                      "PBS_token_ids": t["ids"], "num_blocks": blocks,
                      "attn_output": torch.zeros((case["hq"], case["d"]), device="cuda"),
                      "mean_attn_weights": torch.zeros(dense + blocks * case["kgs"], device="cuda")})
    return {"case": case, "batch": batch}


def _run_batched(s):
    case = s["case"]
    _C.fused_attention_decode_batched(s["batch"], case["hq"], case["hkv"], case["d"], case["kgs"], case["meta"])
    return [[e["attn_output"], e["mean_attn_weights"]] for e in s["batch"]]


# ---------------------------------------------------------------------------
# Engine
# ---------------------------------------------------------------------------
def _cache(case, room):
    return TriTierCache(case["prompt"] + room, case["d"], case["hkv"], RECENT, HEAVY, num_q_heads=case["hq"],
                        k_group_size=case["kgs"], pbs_metadata_dtype=case["meta"])


def _prompt(g, case):
    n, h, d = case["prompt"], case["hkv"], case["d"]
    return _keys(g, n, h, d), _values(g, n, h, d)


def _token(g, case):
    q = torch.randn(case["hq"] * case["d"], generator=g, device="cuda")
    k, v = (torch.randn(case["hkv"] * case["d"], generator=g, device="cuda") for _ in range(2))
    return q, k, v


_ROOM = 16384  # decode tokens an engine case has room for


def _prepare_engine(case, seed):
    g = _generator(seed)
    s = {"case": case, "caches": [], "tokens": [],
         "out": torch.zeros((case["layers"], case["hq"] * case["d"]), device="cuda")}
    for _ in range(case["layers"]):
        cache = _cache(case, _ROOM)
        k, v = _prompt(g, case)
        cache.prefill(k, v)
        torch.cuda.synchronize()  # the prompt's memory is given back here
        s["caches"].append(cache)
        s["tokens"].append(_token(g, case))
    return s


def _run_engine(s):
    """One decode token through the layers."""
    prev = s["caches"][-1] if len(s["caches"]) > 1 else None
    for i, (cache, (q, k, v)) in enumerate(zip(s["caches"], s["tokens"])):
        if s["case"]["deferred"]:
            cache.step_deferred(q, k, v, s["out"][i], prev=prev)
            prev = cache
        else:
            cache.step(q, k, v, s["out"][i])
    return [s["out"], [c.Global_Attn_Scr for c in s["caches"]], [c.HH_token_ids for c in s["caches"]]]


def _prepare_prefill(case, seed):
    g = _generator(seed)
    k, v = _prompt(g, case)
    return {"case": case, "k": k, "v": v, "token": _token(g, case)}


def _run_prefill(s):
    s["cache"] = cache = _cache(s["case"], 4096)
    cache.prefill(s["k"], s["v"])
    out = torch.empty(s["case"]["hq"] * s["case"]["d"], device="cuda")
    cache.step(*s["token"], out)
    return [out, cache.Global_Attn_Scr, cache.S_K_Buffer, cache.S_V_Buffer, cache.RW_K_Buffer, cache.RW_V_Buffer,
            cache.HH_token_ids, cache.WR_token_ids]


# ---------------------------------------------------------------------------
# Quantise and dequantise
# ---------------------------------------------------------------------------
def _prepare_quantize(case, seed):
    g = _generator(seed)
    nb, h, d, kgs = case["blocks"], case["h"], case["d"], case["kgs"]
    n, meta = nb * kgs, torch.uint16 if case["meta"] == "fp16" else torch.float32
    empty = lambda shape, t: torch.empty(shape, dtype=t, device="cuda")  # noqa: E731
    return {"case": case, "k": _keys(g, n, h, d), "v": _values(g, n, h, d),
            "kp": empty((nb, kgs // 16, h, d), torch.int32), "ks": empty((nb, h, d), meta),
            "kz": empty((nb, h, d), meta), "vp": empty((n, h, d // 16), torch.int32), "vs": empty((n, h), meta),
            "vz": empty((n, h), meta)}


def _run_quantize(s):
    c = s["case"]
    _C.quantize_k_blocks(s["k"], s["kp"], s["ks"], s["kz"], c["blocks"], c["h"], c["d"], c["kgs"], c["meta"])
    _C.quantize_v_block(s["v"], s["vp"], s["vs"], s["vz"], c["h"], c["d"], c["blocks"] * c["kgs"], c["meta"])
    return [_bits(s[k]) for k in ("kp", "ks", "kz", "vp", "vs", "vz")]


def _bits(t):
    return t.view(torch.int16) if t.dtype == torch.uint16 else t


def _prepare_dequantize(case, seed):
    g = _generator(seed)
    nb, h, d, kgs = case["blocks"], case["h"], case["d"], case["kgs"]
    s = _pbs(g, {"hkv": h, "d": d, "kgs": kgs, "meta": case["meta"]}, nb)
    return {"case": case, **s, "k": torch.empty((nb * kgs, h, d), device="cuda"),
            "v": torch.empty((nb * kgs, h, d), device="cuda")}


def _run_dequantize(s):
    c = s["case"]
    _C.dequantize_k(s["kp"], s["ks"], s["kz"], s["k"], c["blocks"], c["h"], c["d"], c["kgs"], c["meta"])
    _C.dequantize_v(s["vp"], s["vs"], s["vz"], s["v"], c["blocks"] * c["kgs"], c["h"], c["d"], c["meta"])
    return [s["k"], s["v"]]


# ---------------------------------------------------------------------------
# Entry points
# ---------------------------------------------------------------------------
_PREPARE = {"attention": _prepare_attention, "batched": _prepare_batched, "engine": _prepare_engine,
            "prefill": _prepare_prefill, "quantize": _prepare_quantize, "dequantize": _prepare_dequantize}
_RUN = {"attention": _run_attention, "batched": _run_batched, "engine": _run_engine, "prefill": _run_prefill,
        "quantize": _run_quantize, "dequantize": _run_dequantize}


def prepare(case, seed):
    return _PREPARE[case["kind"]](case, seed)


def run(state):
    return _RUN[state["case"]["kind"]](state)


def _packed_bytes(h, d, blocks, kgs, meta):
    m, n = 2 if meta == "fp16" else 4, blocks * kgs
    return n // 16 * h * d * 4 + blocks * h * d * 2 * m + n * h * (d // 16) * 4 + n * h * 2 * m


def _step_work(case, dense, blocks, weights=True):
    """Bytes and operations of one decode attention: query, tiers, token ids, output and mean weights once."""
    hq, hkv, d, kgs = case["hq"], case["hkv"], case["d"], case["kgs"]
    n = dense + blocks * kgs
    b = 2 * hq * d * 4 + 2 * dense * hkv * d * 4 + _packed_bytes(hkv, d, blocks, kgs, case["meta"]) + blocks * kgs * 8
    return b + (n * 4 if weights else 0), 4.0 * hq * d * n


def _prompt_blocks(case):
    return (case["prompt"] - SINK - RECENT) // case["kgs"]


def work(case):
    kind = case["kind"]
    if kind == "attention":
        b, f = _step_work(case, case["dense"], case["blocks"], case["weights"])
        return {"bytes": case["layers"] * b, "flops": case["layers"] * f}
    if kind == "batched":
        w = [_step_work(case, *_blocks_of(case, t)[:2]) for t in _lengths(case)]
        return {"bytes": sum(b for b, _ in w), "flops": sum(f for _, f in w)}
    if kind == "engine":
        b, f = _step_work(case, SINK + RECENT + 1, _prompt_blocks(case))
        b += 4 * case["hkv"] * case["d"] * 4 * 2  # the new token in, the evicted one out of the ring and into its tier
        return {"bytes": case["layers"] * b, "flops": case["layers"] * f}
    if kind == "prefill":
        b, f = _step_work(case, SINK + RECENT + 1, _prompt_blocks(case))
        rows = case["prompt"] - _prompt_blocks(case) * case["kgs"]
        row = 2 * case["hkv"] * case["d"] * 4
        packed = _packed_bytes(case["hkv"], case["d"], _prompt_blocks(case), case["kgs"], case["meta"])
        return {"bytes": b + (case["prompt"] + rows) * row + packed, "flops": f + 10.0 * case["prompt"] * row / 4}
    n = 2 * case["blocks"] * case["kgs"] * case["h"] * case["d"]
    b = 4 * n + _packed_bytes(case["h"], case["d"], case["blocks"], case["kgs"], case["meta"])
    return {"bytes": b, "flops": (5.0 if kind == "quantize" else 2.0) * n}


def tolerance(case):
    # Packed words, scales and zeros, and the rounded fma of the dequantisers are fixed bit for bit.
    if case["kind"] in ("quantize", "dequantize"):
        return "exact"
    # FP32 sums in another order and one hardware exponential per weight: outputs and mean weights within a few
    # 1e-7 (2-norm) of 64-bit attention over the same tiers; single mean weights of a long context, each a sum
    # over the heads of 2^(logit), differ by a few 1e-6.
    return {"rel": 4e-6, "max": 1e-4}


# ---------------------------------------------------------------------------
# 64-bit results
# ---------------------------------------------------------------------------
def _meta64(t):
    return (t.view(torch.float16) if t.dtype == torch.uint16 else t).double()


def _codes(words, dim):
    shift = 2 * torch.arange(16, device=words.device, dtype=torch.int32)
    shift = shift.view([16 if i == dim else 1 for i in range(words.dim() + 1)])
    return (words.unsqueeze(dim) >> shift) & 3


def _unpack_keys(kp, ks, kz, kgs):
    nb, _, h, d = kp.shape
    q = _codes(kp, 2).view(nb, kgs, h, d).double()
    return (q * _meta64(ks)[:, None] + _meta64(kz)[:, None]).view(nb * kgs, h, d)


def _unpack_values(vp, vs, vz):
    n, h, w = vp.shape
    q = _codes(vp, 3).reshape(n, h, 16 * w).double()
    return q * _meta64(vs)[..., None] + _meta64(vz)[..., None]


def _attend64(q, k, v, masked_ids=None, dense=0):
    """Output [Hq, D] and mean weights [N] of 64-bit softmax attention; q [Hq, D], k and v [N, Hkv, D]."""
    hq, d = q.shape
    hkv = k.shape[1]
    qh = q.double().view(hkv, hq // hkv, d)
    s = torch.matmul(qh, k.permute(1, 2, 0).contiguous()) / math.sqrt(d)
    if masked_ids is not None and masked_ids.numel():
        s[:, :, dense:].masked_fill_(masked_ids == -1, -math.inf)
    w = torch.softmax(s, -1)
    out = torch.matmul(w, v.permute(1, 0, 2).contiguous())
    return out.reshape(hq, d), w.reshape(hq, -1).mean(0)


def _sequence64(t, kgs):
    k, v = t["dk"].double(), t["dv"].double()
    if t["kp"].shape[0]:
        k = torch.cat([k, _unpack_keys(t["kp"], t["ks"], t["kz"], kgs)])
        v = torch.cat([v, _unpack_values(t["vp"], t["vs"], t["vz"])])
    return _attend64(t["q"], k, v, t["ids"], t["dk"].shape[0])


def _first_step64(case, k, v, token, length):
    """Output and scores [length] of the first decode step after a prompt: its oldest recent token became the first
    heavy hitter (all scores are still zero), the sinks, the recent window and the new token are in FP32, the whole
    blocks between are packed and the tokens left over wait, not attended."""
    h, d, n, kgs = case["hkv"], case["d"], case["prompt"], case["kgs"]
    q, kn, vn = token
    q, kn, vn = q.view(-1, d), kn.view(1, h, d), vn.view(1, h, d)
    ids = torch.arange(n + 1, device="cuda")
    m = _prompt_blocks(case) * kgs
    keep = torch.cat([ids[:SINK + m], ids[n - RECENT:]])
    parts = [torch.cat([x[:SINK].double(), y, x[n - RECENT:].double(), z.double()]) for x, y, z in (
        (k, _unpack_keys(*_pack_keys(k[SINK:SINK + m], kgs, case["meta"]), kgs), kn),
        (v, _unpack_values(*_pack_values(v[SINK:SINK + m], case["meta"])), vn))]
    out, w = _attend64(q, *parts)
    g = torch.zeros(length, dtype=torch.float64, device="cuda")
    g[keep] = w
    return out.reshape(-1), g


def exact(case, seed):
    kind = case["kind"]
    g = _generator(seed)
    if kind == "attention":
        got = []
        for _ in range(case["layers"]):
            got.append(_sequence64(_sequence(g, case, case["dense"], case["blocks"], case["masked"]), case["kgs"]))
        out = [torch.stack([o for o, _ in got]), torch.stack([m for _, m in got])]
        return out if case["weights"] else out[:1]
    if kind == "batched":
        return [list(_sequence64(_sequence(g, case, *_blocks_of(case, t)), case["kgs"])) for t in _lengths(case)]
    if kind == "engine":
        outs, scores = [], []
        for i in range(case["layers"]):
            k, v = _prompt(g, case)
            o, w = _first_step64(case, k, v, _token(g, case), case["prompt"] + _ROOM)
            outs.append(o)
            # a deferred step leaves the last layer's feedback for the next token
            scores.append(torch.zeros_like(w) if case["deferred"] and i == case["layers"] - 1 else w)
        return [torch.stack(outs), scores, [None] * case["layers"]]
    if kind == "prefill":
        k, v = _prompt(g, case)
        o, w = _first_step64(case, k, v, _token(g, case), case["prompt"] + 4096)
        return [o, w, None, None, None, None, None, None]
    if kind == "dequantize":
        s = _pbs(g, {"hkv": case["h"], "d": case["d"], "kgs": case["kgs"], "meta": case["meta"]}, case["blocks"])
        return [_unpack_keys(s["kp"], s["ks"], s["kz"], case["kgs"]), _unpack_values(s["vp"], s["vs"], s["vz"])]
    if case["meta"] == "fp16":
        return None  # whole numbers only
    k = _keys(g, case["blocks"] * case["kgs"], case["h"], case["d"]).double()
    v = _values(g, case["blocks"] * case["kgs"], case["h"], case["d"]).double()
    x = k.view(case["blocks"], case["kgs"], case["h"], case["d"])
    return [None, ((x.amax(1) - x.amin(1)) / 3).clamp_min(1e-9), x.amin(1), None,
            ((v.amax(2) - v.amin(2)) / 3).clamp_min(1e-9), v.amin(2)]
