"""Performance cases of the framework's two operators: paged decode attention
and the fused RoPE + paged K/V write, through their public entry points.

Decode cases run either the torch operator (``attnarc_amd.torch_ops``, what a
torch program binds: native NHD caches, the output allocated by the call) or
the extended operator (``attnarc_amd.ops``: FP8 caches, HND layout, log-sum-exp
output, a partition size chosen by the caller, who keeps the output and the
split-K workspace). Write cases run ``rope_paged_kv_write_`` on column slices
of one packed QKV projection. Caches, block tables and slots are shuffled as a
serving pool's are. A case holds plain sizes; its sequence lengths are spread
evenly between ``ctx_min`` and ``ctx_max``, in an order the seed decides.
"""

from __future__ import annotations

import math

import numpy as np
import torch

from attnarc_amd import ops, torch_ops, workloads

_DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
_BYTES = {"f32": 4, "f16": 2, "bf16": 2}
_DEVICE = "cuda:0"


def _decode(name, entry, dtype, kv, layout, batch, heads, head_size, ctx, partition=0, block_size=16, lse=False):
    case = {"op": "decode", "entry": entry, "dtype": dtype, "kv": kv, "layout": layout, "batch": batch,
            "query_heads": heads[0], "kv_heads": heads[1], "head_size": head_size, "block_size": block_size,
            "ctx_min": ctx[0], "ctx_max": ctx[1], "partition": partition, "lse": lse}
    return {"name": name, **case} if name else case


def _write(name, dtype, kv, layout, tokens, heads, head_size, rotary, neox=True, block_size=16):
    case = {"op": "rope", "dtype": dtype, "kv": kv, "layout": layout, "tokens": tokens, "query_heads": heads[0],
            "kv_heads": heads[1], "head_size": head_size, "rotary": rotary, "neox": neox, "block_size": block_size}
    return {"name": name, **case} if name else case


def listed():
    return [
        # One user's first tokens: a single short sequence, where launches and latency count.
        _decode("op_b1_ctx128", "torch", "bf16", "native", "NHD", 1, (32, 8), 128, (128, 128)),
        # A small serving batch over one interleaved K/V cache, F16.
        _decode("op_b8_ctx1024_interleaved", "torch", "f16", "native", "interleaved", 8, (32, 8), 128, (993, 1024)),
        # F32 multi-head attention of a tiny model under test.
        _decode("f32_mha_d64_small", "extended", "f32", "native", "NHD", 4, (8, 8), 64, (1, 256)),
        # A mid-sized batch of a small GQA model at one context length, no partitions asked for.
        _decode("gqa12x2_b32_ctx2048", "extended", "bf16", "native", "NHD", 32, (12, 2), 128, (2048, 2048)),
        # The serving batch of an 8B GQA model: ragged contexts, 512-token partitions.
        _decode("gqa32x8_b64_ragged8k", "extended", "bf16", "native", "NHD", 64, (32, 8), 128, (512, 8192), 512),
        # A large batch of a 70B GQA model over an FP8 cache in HND order.
        _decode("gqa64x8_b128_fp8_hnd", "extended", "bf16", "fp8", "HND", 128, (64, 8), 128, (4096, 4096), 512),
        # Long documents under multi-query attention.
        _decode("mqa32_b8_ctx128k", "extended", "bf16", "native", "NHD", 8, (32, 1), 128, (65536, 131072), 1024),
        # A model evaluated in F32: grouped heads, ragged contexts, log-sum-exp wanted.
        _decode("f32_gqa32x8_ragged4k", "extended", "f32", "native", "NHD", 16, (32, 8), 128, (255, 4093), 512,
                lse=True),
        # Multi-head attention of head size 96 over an FP8 cache, ragged.
        _decode("mha32_d96_fp8_ragged", "extended", "bf16", "fp8", "NHD", 32, (32, 32), 96, (301, 4001), 512),
        # A wide multi-query group over an FP8 cache.
        _decode("mqa48_fp8_ctx16k", "extended", "bf16", "fp8", "NHD", 64, (48, 1), 128, (8193, 16384), 512),
        # The K/V write of one decode step of a serving batch into an FP8 cache.
        _write("write_step61_fp8", "bf16", "fp8", "HND", 61, (32, 8), 128, 128),
        # The K/V write of a large prefill chunk.
        _write("write_prefill32k", "bf16", "native", "NHD", 32768, (32, 8), 128, 128),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


_MAX_KV_BYTES = 1.2e9  # about the largest listed case's


def _fit(batch, heads, head_size, elem, ctx_max):
    """The largest batch up to ``batch`` whose K/V stays within _MAX_KV_BYTES."""
    return max(1, min(batch, int(_MAX_KV_BYTES / (ctx_max * heads[1] * head_size * 2 * elem))))


def draw(rng):
    kind = rng.choice(["torch", "serve", "serve", "fp8", "fp8", "f32", "long", "wide", "write", "write"])
    if kind == "torch":  # short contexts through the torch operator
        heads = rng.choice([(32, 8), (12, 2), (8, 8), (28, 4), (40, 8)])
        ctx = _log(rng, 16, 4096)
        return _decode(None, "torch", rng.choice(["bf16", "f16"]), "native", rng.choice(["NHD", "interleaved"]),
                       _log(rng, 1, 64), heads, rng.choice([64, 128]), (max(1, ctx - rng.choice([0, 31])), ctx))
    if kind in ("serve", "fp8"):  # serving batches, native or FP8 caches, every head size served
        heads = rng.choice([(32, 8), (64, 8), (16, 8), (12, 2), (32, 32), (20, 20), (24, 4), (32, 4)])
        head_size = rng.choice([64, 80, 96, 112, 128, 128, 256])
        kv = "fp8" if kind == "fp8" else "native"
        ctx_max = _log(rng, 700, 16384)
        batch = _fit(_log(rng, 4, 160), heads, head_size, 1 if kv == "fp8" else 2, ctx_max)
        ctx_min = rng.choice([ctx_max, ctx_max // 2, ctx_max // 16])
        return _decode(None, "extended", rng.choice(["bf16", "bf16", "f16"]), kv, rng.choice(["NHD", "HND"]), batch,
                       heads, head_size, (ctx_min, ctx_max), rng.choice([0, 256, 512, 512]),
                       rng.choice([16, 16, 32, 64]), rng.random() < 0.25)
    if kind == "f32":
        heads = rng.choice([(8, 8), (32, 8), (12, 2), (16, 8)])
        head_size = rng.choice([64, 80, 128])
        ctx_max = _log(rng, 64, 4096)
        batch = _fit(_log(rng, 2, 32), heads, head_size, 4, ctx_max)
        return _decode(None, "extended", "f32", "native", rng.choice(["NHD", "HND"]), batch, heads, head_size,
                       (max(1, ctx_max // 16), ctx_max), rng.choice([0, 512]) if ctx_max > 512 else 0, 16,
                       rng.random() < 0.5)
    if kind == "long":  # few long sequences
        heads = rng.choice([(32, 1), (16, 1), (32, 8), (24, 2)])
        kv = rng.choice(["native", "native", "fp8"])
        ctx_max = _log(rng, 16384, 131072)
        batch = _fit(_log(rng, 1, 12), heads, 128, 1 if kv == "fp8" else 2, ctx_max)
        return _decode(None, "extended", "bf16", kv, "NHD", batch, heads, 128, (ctx_max // 2, ctx_max), 1024)
    if kind == "wide":  # wide multi-query groups
        heads, head_size = rng.choice([((48, 1), 128), ((64, 1), 128), ((71, 1), 64), ((24, 1), 64), ((128, 1), 128)])
        kv = rng.choice(["native", "fp8"])
        ctx_max = _log(rng, 1024, 16384)
        batch = _fit(_log(rng, 8, 64), heads, head_size, 1 if kv == "fp8" else 2, ctx_max)
        return _decode(None, "extended", rng.choice(["bf16", "f16"]), kv, "NHD", batch, heads, head_size,
                       (ctx_max // 2, ctx_max), 512)
    # K/V writes from a decode step to a prefill chunk
    heads = rng.choice([(32, 8), (64, 8), (12, 2), (32, 32), (32, 1)])
    head_size = rng.choice([64, 80, 96, 128, 128, 256])
    dtype = rng.choice(["bf16", "bf16", "f16", "f32"])
    row = (heads[0] + 2 * heads[1]) * head_size * _BYTES[dtype]
    tokens = min(_log(rng, 1, 32768), int(4.5e8 / row))
    rotary = head_size if rng.random() < 0.75 else head_size // 2
    return _write(None, dtype, rng.choice(["native", "fp8"]), rng.choice(["NHD", "HND"]), tokens, heads, head_size,
                  rotary, rng.random() < 0.75, rng.choice([16, 16, 32]))


def _lengths(case):
    b = case["batch"]
    if b == 1:
        return [case["ctx_max"]]
    return [int(round(x)) for x in np.linspace(case["ctx_min"], case["ctx_max"], b)]


def _prepare_decode(case, seed):
    lengths = _lengths(case)
    np.random.default_rng(seed).shuffle(lengths)
    interleaved = case["layout"] == "interleaved"
    fixed = case["ctx_min"] == case["ctx_max"]
    w = workloads.make_case(
        name="decode", dtype=_DTYPES[case["dtype"]], sequences=case["batch"], query_heads=case["query_heads"],
        kv_heads=case["kv_heads"], head_size=case["head_size"], value_head_size=case["head_size"],
        block_size=case["block_size"], lengths=lengths, seed=seed, device=_DEVICE, cache_encoding=case["kv"],
        layout="NHD" if interleaved else case["layout"], pool_factor=None if fixed else 1.25,
        partition_tokens=case["partition"])
    state = {"case": case, "workload": w}
    if interleaved:
        state["kv_cache"] = torch.stack((w.key_cache, w.value_cache), dim=1)
        w.key_cache, w.value_cache = state["kv_cache"][:, 0], state["kv_cache"][:, 1]
    if case["entry"] == "extended":
        state["output"] = torch.empty_like(w.query)
        state["lse"] = torch.empty(w.query.shape[:2], device=_DEVICE) if case["lse"] else None
        need = ops.extended_workspace_elements(w.sequences, w.query_heads, w.value_head_size, w.max_sequence_length,
                                               w.partition_tokens)
        state["workspace"] = torch.empty(need, device=_DEVICE) if need else None
    return state


def _prepare_write(case, seed):
    gen = torch.Generator(device=_DEVICE).manual_seed(seed)
    dtype, t, d, bs = _DTYPES[case["dtype"]], case["tokens"], case["head_size"], case["block_size"]
    hq, hkv, rotary = case["query_heads"], case["kv_heads"], case["rotary"]
    packed = torch.randn((t, (hq + 2 * hkv) * d), generator=gen, device=_DEVICE).to(dtype)
    query, key, value = (x.unflatten(1, (-1, d)) for x in packed.split((hq * d, hkv * d, hkv * d), dim=1))
    max_position = 8192
    inv = 10000.0 ** (-torch.arange(0, rotary, 2, device=_DEVICE, dtype=torch.float64) / rotary)
    angles = torch.arange(max_position, device=_DEVICE, dtype=torch.float64)[:, None] * inv
    num_blocks = -(-5 * t // (4 * bs)) + 1
    slots = torch.randperm(num_blocks, generator=gen, device=_DEVICE)[:, None] * bs
    slots = (slots + torch.arange(bs, device=_DEVICE)).flatten()[:t].contiguous()
    cache_dtype = torch.uint8 if case["kv"] == "fp8" else dtype
    if case["layout"] == "NHD":
        cache = torch.zeros((num_blocks, 2, bs, hkv, d), device=_DEVICE, dtype=cache_dtype)
    else:
        cache = torch.zeros((num_blocks, 2, hkv, bs, d), device=_DEVICE, dtype=cache_dtype).transpose(2, 3)
    scales = torch.rand((2, hkv), generator=gen, device=_DEVICE) * 0.09 + 0.01
    return {
        "case": case, "query": query, "key": key, "value": value,
        "positions": torch.randint(0, max_position, (t,), generator=gen, device=_DEVICE),
        "cos_sin": torch.cat((angles.cos(), angles.sin()), dim=1).to(dtype),
        "kv_cache": cache, "key_scales": scales[0].clone(), "value_scales": scales[1].clone(), "slots": slots,
    }


def prepare(case, seed):
    """What the program holds before the call: caches, tables, queries, and the buffers it keeps."""
    return _prepare_decode(case, seed) if case["op"] == "decode" else _prepare_write(case, seed)


def run(state):
    case = state["case"]
    if case["op"] == "rope":
        return ops.rope_paged_kv_write_(
            state["query"], state["key"], state["value"], state["positions"], state["cos_sin"], state["kv_cache"],
            state["key_scales"], state["value_scales"], state["slots"], case["neox"])
    w = state["workload"]
    if case["entry"] == "torch":
        return torch_ops.paged_decode_attention(
            w.query, w.key_cache, w.value_cache, w.block_tables, w.sequence_lengths,
            max_sequence_length=w.max_sequence_length, scale=w.scale)
    return ops.paged_decode_attention_extended(
        w.query, w.key_cache, w.value_cache, w.block_tables, w.sequence_lengths,
        max_sequence_length=w.max_sequence_length, scale=w.scale, layout=w.layout, key_scales=w.key_scales,
        value_scales=w.value_scales, partition_tokens=w.partition_tokens, output=state["output"], lse=state["lse"],
        return_lse=case["lse"], workspace=state["workspace"])


def work(case):
    e = _BYTES[case["dtype"]]
    ce = 1 if case["kv"] == "fp8" else e
    hq, hkv, d = case["query_heads"], case["kv_heads"], case["head_size"]
    if case["op"] == "rope":
        t, r = case["tokens"], case["rotary"]
        rows = 2 * (hq + hkv) * r + hkv * (d - r) + hkv * d  # rotated dims read and written; K tail and V read
        return {"bytes": t * (rows * e + r * e + 16 + 2 * hkv * d * ce), "flops": t * (hq + hkv) * r * 3}
    tokens, b = sum(_lengths(case)), case["batch"]
    blocks = sum(-(-n // case["block_size"]) for n in _lengths(case))
    return {"bytes": tokens * hkv * 2 * d * ce + b * hq * d * 2 * e + blocks * 4 + b * 4 + (b * hq * 4 if case["lse"] else 0),
            "flops": 4 * tokens * hq * d}


def tolerance(case):
    """About four times the measured distance to 64 bits: the output type's
    rounding for 16-bit types (1.7e-3 BF16, 2.5e-4 F16), and the order of the
    F32 sums (up to 4.3e-7, larger for longer rows) for F32. The write rounds each
    rotated value once, in an order of operations its contract fixes."""
    if case["op"] == "rope":
        return "exact"
    return {"f32": {"rel": 4e-6}, "f16": {"rel": 1e-3}, "bf16": {"rel": 7e-3}}[case["dtype"]]


def _exact_decode(case, seed):
    w = _prepare_decode(case, seed)["workload"]
    hnd = w.layout == "HND"
    group, d = w.query_heads // w.kv_heads, w.head_size
    out = torch.empty(w.query.shape, device=_DEVICE, dtype=torch.float64)
    lse = torch.empty(w.query.shape[:2], device=_DEVICE, dtype=torch.float64)
    for s, length in enumerate(w.lengths):
        blocks = w.block_tables[s, : -(-length // w.block_size)].long()

        def rows(cache, scales):  # [kv_heads, length, dim] in 64 bits
            x = cache[blocks].double()
            x = (x.permute(1, 0, 2, 3) if hnd else x.permute(2, 0, 1, 3)).reshape(w.kv_heads, -1, d)[:, :length]
            return x if scales is None else x * scales.double()[:, None, None]

        q = w.query[s].double().view(w.kv_heads, group, d)
        k = rows(w.key_cache, w.key_scales).transpose(1, 2).contiguous()
        scores = torch.matmul(q, k) * w.scale
        lse[s] = torch.logsumexp(scores, dim=-1).flatten()
        out[s] = torch.matmul(torch.softmax(scores, dim=-1), rows(w.value_cache, w.value_scales).contiguous()).view(-1, d)
    return (out, lse) if case["lse"] else out


def _exact_write(case, seed):
    s = _prepare_write(case, seed)
    rotary = case["rotary"]
    cos, sin = s["cos_sin"][s["positions"]].double().chunk(2, dim=1)

    def rotate(x):
        y = x.double()
        if case["neox"]:
            a, b = y[..., : rotary // 2], y[..., rotary // 2 : rotary]
        else:
            a, b = y[..., 0:rotary:2], y[..., 1:rotary:2]
        c, n = cos[:, None], sin[:, None]
        ra, rb = a * c - b * n, b * c + a * n
        rotated = torch.cat((ra, rb), dim=-1) if case["neox"] else torch.stack((ra, rb), dim=-1).flatten(-2)
        return torch.cat((rotated, y[..., rotary:]), dim=-1)

    query, key = rotate(s["query"]), rotate(s["key"])
    if case["kv"] == "fp8":  # the cache holds codes
        return query, key, None
    cache = s["kv_cache"].double()
    block, page = s["slots"] // case["block_size"], s["slots"] % case["block_size"]
    cache[block, 0, page] = key
    cache[block, 1, page] = s["value"].double()
    return query, key, cache


def exact(case, seed):
    return _exact_decode(case, seed) if case["op"] == "decode" else _exact_write(case, seed)
