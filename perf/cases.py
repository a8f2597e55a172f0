"""
The workloads whose speed this library answers for, as its users run them, each through the public entry points:

``sdpa``      ``HipSDPA.scaled_dot_product_attention``: a chunk of queries (or one) over a cache that the caller holds,
              with the per-key score-sums that the eviction policies live on; plain, 8-bit and 4-bit stores.
``decode``    ``H2OKVCache.forward`` with one new token per sequence and a full cache: slot write, attention, score
              update, choice of the next slot. What a generation loop calls once per layer and token.
``chunk``     the same with a chunk of tokens: what a long prompt goes through once the cache is full.
``prompt``    the first chunk of a sequence into an empty cache: causal attention and the write of all rows.
``quantize``  ``RowQuantizer``: a store's rows to codes and back.
``model``     ``LongContextPrefillModel.prefill``: a prompt in chunks through a decoder stack over H2O caches.

A case is a dict of plain values. Shapes are the ones of the benchmark's configurations (an attention layer of 8 / 2
heads of 64; 32 / 8 heads of 128 with caches of 16384 to 131072 slots, chunks of 1024, batch 1 and 8), of the tests
(ragged lengths, 1 to 8 heads per KV head, head sizes 64, 128 and 256, float16 rows) and what lies between them.
"""
import dataclasses
import math

import torch

from keys_values_amd.attention import ops
from keys_values_amd.attention.sdpa import HipSDPA
from keys_values_amd.kvcache.h2o import KVCacheParams, create_kv_cache
from keys_values_amd.kvcache.quantize import RowQuantizer
from keys_values_amd.longctx.model import QWEN3_4B, LongContextPrefillModel

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}
BITS = {"plain": 16, "u8": 8, "u4": 4}
STORES = {"plain": "default", "u8": "torch-quantized8", "u4": "torch-quantized4"}
HEADS = [(32, 8), (32, 8), (8, 2), (28, 4), (24, 8), (32, 4), (16, 8), (8, 8)]  # query heads / KV heads
CHUNK_STEPS_BEFORE = 3  # chunk steps between the prompt and the measured ones: the slots are scattered by then


def _sdpa(name, B, heads, D, q, T, dtype="bf16", store="plain", scattered=False, weights=True):
    return {"name": name, "kind": "sdpa", "B": B, "Hq": heads[0], "Hkv": heads[1], "D": D, "q": q, "T": T, "dtype": dtype,
            "store": store, "scattered": scattered, "weights": weights}


def _cache(name, kind, B, heads, D, q, T, dtype="bf16", store="plain", policy="h2o", grace=0, normalize=False):
    return {"name": name, "kind": kind, "B": B, "Hq": heads[0], "Hkv": heads[1], "D": D, "q": q, "T": T, "dtype": dtype,
            "store": store, "policy": policy, "grace": grace, "normalize": normalize}


def listed():
    return [
        # one attention layer at the smallest configuration: launches and host work count
        _sdpa("sdpa_small", 1, (8, 2), 64, 128, 1024),
        # a batch of two, seven heads per KV head, nothing a multiple of a tile, slots in the order an evicting cache leaves
        _sdpa("sdpa_ragged", 2, (28, 4), 128, 333, 5001, dtype="fp16", scattered=True),
        # the benchmark's headline: a 1024-token chunk at the end of 32768 positions
        _sdpa("sdpa_large", 1, (32, 8), 128, 1024, 32768),
        # the same over a quantised store of 65536 positions
        _sdpa("sdpa_u8_large", 1, (32, 8), 128, 1024, 65536, store="u8"),
        # generation for one user with a small cache: one call per layer and token, latency is everything
        _cache("decode_small", "decode", 1, (32, 8), 128, 1, 4096),
        # a serving batch over 8-bit caches of 16384 slots with a ring of recent tokens
        _cache("decode_u8", "decode", 4, (32, 8), 128, 1, 16384, store="u8", grace=64),
        # the benchmark's decode configuration: 8 sequences, 131072 slots each
        _cache("decode_large", "decode", 8, (32, 8), 128, 1, 131072),
        # one layer's share of the long-context configuration: a 1024-token chunk into 16384 8-bit slots
        _cache("chunk_u8", "chunk", 1, (32, 8), 128, 1024, 16384, store="u8"),
        # the heaviest eviction policy on a short odd-sized chunk
        _cache("chunk_policy", "chunk", 2, (24, 8), 128, 200, 6000, store="u8", policy="qh2o-vlen", grace=128, normalize=True),
        # the first chunk of a long prompt
        _cache("prompt_long", "prompt", 1, (32, 8), 128, 8192, 16384, store="u8"),
        # one tensor of a 65536-slot store to codes and back
        {"name": "quantize_store", "kind": "quantize", "B": 1, "Hkv": 8, "D": 128, "T": 65536, "start": 0, "end": 65536, "bits": 8,
         "over_heads": False, "dtype": "bf16"},
        # two layers of the long-context stack: a 4096-token first chunk, then chunks of 1024
        {"name": "model_prefill", "kind": "model", "layers": 2, "T": 4096, "chunk": 1024, "tokens": 8192, "store": "u8"},
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _some_size(rng, low, high):
    """A size of [low, high], even over its logarithm: a power of two, a multiple of 64 or any number."""
    n = _log_int(rng, low, high)
    how = rng.random()
    if how < 0.25:
        n = 1 << round(math.log2(n))
    elif how < 0.5:
        n = (n + 32) // 64 * 64
    return max(low, min(high, n))


def draw(rng):
    """One more case of the same ranges; no more work than the largest of the listed ones."""
    while True:
        case = _draw(rng)
        w = work(case)
        if w["bytes"] <= 4.4e9 and w["flops"] <= 1.1e12 * (4 if case["kind"] == "model" else 1):
            return case


def _draw(rng):
    kind = rng.choices(["sdpa", "decode", "chunk", "prompt", "quantize", "model"], [30, 27, 20, 9, 9, 5])[0]
    if kind == "quantize":
        heads = rng.choice([2, 4, 8])
        T = _some_size(rng, 256, 65536)
        start = rng.choice([0, 0, rng.randrange(T // 2)])
        end = T if start == 0 else rng.randint(start + 1, T)
        return {"kind": kind, "B": rng.choice([1, 1, 2, 4]), "Hkv": heads, "D": rng.choice([64, 128, 128, 256]), "T": T, "start": start, "end": end,
                "bits": rng.choice([8, 8, 4]), "over_heads": rng.random() < 0.25, "dtype": rng.choice(["bf16", "bf16", "fp16"])}
    if kind == "model":
        T = _some_size(rng, 1024, 8192)
        return {"kind": kind, "layers": rng.choice([1, 2]), "T": T, "chunk": _some_size(rng, 128, min(1024, T // 2)), "tokens": _some_size(rng, T, 2 * T),
                "store": rng.choice(["plain", "u8"])}
    heads = rng.choice(HEADS)
    D = rng.choice([64, 128, 128, 128, 256])
    dtype = rng.choice(["bf16", "bf16", "bf16", "fp16"])
    store = rng.choice(["plain", "plain", "u8", "u4"])
    if kind == "sdpa":
        T = _some_size(rng, 256, 65536)
        q = rng.choice([1, _some_size(rng, 2, min(1024, T // 2)), _some_size(rng, 2, min(1024, T // 2))])
        case = _sdpa("", rng.choice([1, 1, 2, 4]), heads, D, q, T, dtype, store, rng.random() < 0.5, rng.random() < 0.8)
    else:
        policy = rng.choice(["h2o", "h2o", "h2o", "h2o-vlen", "qh2o", "qh2o-vlen"])
        if policy.startswith("qh2o") and store == "plain":
            store = "u8"
        T = _some_size(rng, 512, {"decode": 65536, "chunk": 32768, "prompt": 16384}[kind])
        B = rng.choice([1, 2, 4, 8] if kind == "decode" else [1, 1, 2])
        q = {"decode": 1, "chunk": _some_size(rng, 16, min(1024, T // 4)), "prompt": _some_size(rng, T // 8, T)}[kind]
        grace = rng.choice([0, 0, _some_size(rng, 16, T // 8)])
        case = _cache("", kind, B, heads, D, q, T, dtype, store, policy, grace, rng.random() < 0.25)
    del case["name"]
    return case


# -- inputs ---------------------------------------------------------------------------------------------------


def _randn(gen, *shape, dtype):
    return torch.randn(shape, generator=gen, device="cuda", dtype=dtype)


def _keys(gen, *shape, dtype):
    """Keys as a model produces them: unit variance with one value in a hundred eight times as large."""
    x = _randn(gen, *shape, dtype=dtype)
    return x.mul_(torch.where(torch.rand(shape, generator=gen, device="cuda", dtype=dtype) < 0.01, 8.0, 1.0))


def _positions(gen, B, Hkv, T, q):
    """Token positions of a cache that has evicted for a while, every KV head its own: the chunk's ``q`` positions
    and distinct older ones, in no order. Returns them and the chunk's first position."""
    n_old, input_pos = T - q, 2 * T
    old = 2 * torch.arange(n_old, device="cuda") + torch.randint(0, 2, (B, Hkv, n_old), generator=gen, device="cuda")
    new = torch.arange(input_pos, input_pos + q, device="cuda").expand(B, Hkv, q)
    order = torch.rand((B, Hkv, T), generator=gen, device="cuda").argsort(-1)
    return torch.cat((old, new), -1).gather(-1, order).to(torch.int32), input_pos


def _prepare_sdpa(c, gen):
    B, Hkv, T, D, q, dtype = c["B"], c["Hkv"], c["T"], c["D"], c["q"], DTYPES[c["dtype"]]
    query = _randn(gen, B, c["Hq"], q, D, dtype=dtype)
    key, value = _keys(gen, B, Hkv, T, D, dtype=dtype), _randn(gen, B, Hkv, T, D, dtype=dtype)
    quant = None
    if c["store"] != "plain":
        rows = []
        for x in (key, value):
            qz = RowQuantizer((B, Hkv, T, D), dtype, BITS[c["store"]], allocate_buffers=True, device=x.device)
            qz.quantize(0, T, x)
            rows.append((qz.quant_buffer.view(B, Hkv, T, -1), qz.quant_scales.view(B, Hkv, T), qz.quant_zero_points.view(B, Hkv, T)))
        (key, k_scale, k_zp), (value, v_scale, v_zp) = rows
        quant = ops.QuantState(k_scale, k_zp, v_scale, v_zp)
    positions, input_pos = _positions(gen, B, Hkv, T, q) if c["scattered"] else (None, T - q)
    return {"op": HipSDPA(), "query": query, "key": key, "value": value, "quant": quant, "positions": positions, "input_pos": input_pos,
            "weights": c["weights"]}


def _prepare_cache(c, gen):
    B, Hq, Hkv, T, D, q, dtype = c["B"], c["Hq"], c["Hkv"], c["T"], c["D"], c["q"], DTYPES[c["dtype"]]
    chunk = q if c["kind"] == "chunk" else min(256, T // 4)
    cache = create_kv_cache(f"{c['policy']}-{STORES[c['store']]}", KVCacheParams(B, Hkv, T, D, Hq, dtype), max_chunk_size=chunk,
                            normalize_scores=c["normalize"], grace_period=c["grace"])

    def tokens(n):
        return _randn(gen, B, Hq, n, D, dtype=dtype), _keys(gen, B, Hkv, n, D, dtype=dtype), _randn(gen, B, Hkv, n, D, dtype=dtype)

    if c["kind"] != "prompt":  # a prompt that fills the cache, then chunks until the slots are scattered
        cache.forward(*tokens(T))
        for _ in range(CHUNK_STEPS_BEFORE):
            cache.forward(*tokens(chunk))
    return {"cache": cache, "tokens": tokens(q)}


def _prepare_quantize(c, gen):
    dtype = DTYPES[c["dtype"]]
    qz = RowQuantizer((c["B"], c["Hkv"], c["T"], c["D"]), dtype, c["bits"], c["over_heads"], allocate_buffers=True)
    # the slots outside the range hold codes too, as in a store in use
    qz.quant_buffer.fill_(7)
    return {"quantizer": qz, "rows": _keys(gen, c["B"], c["Hkv"], c["end"] - c["start"], c["D"], dtype=dtype), "range": (c["start"], c["end"])}


def _prepare_model(c, gen, seed):
    cfg = dataclasses.replace(QWEN3_4B, n_layer=c["layers"], vocab_size=32768)
    model = LongContextPrefillModel(cfg, cache_length=c["T"], chunk_size=c["chunk"], quantized=c["store"] == "u8", max_context=16384, seed=seed)
    return {"model": model, "ids": torch.randint(0, cfg.vocab_size, (1, c["tokens"]), generator=gen, device="cuda")}


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    kind = case["kind"]
    if kind == "sdpa":
        state = _prepare_sdpa(case, gen)
    elif kind == "quantize":
        state = _prepare_quantize(case, gen)
    elif kind == "model":
        state = _prepare_model(case, gen, seed)
    else:
        state = _prepare_cache(case, gen)
    state["kind"] = kind
    return state


# -- one pass -------------------------------------------------------------------------------------------------


def _bits(t):
    """Stored rows and their states as bit patterns: they are written once and not computed with."""
    return t if t.dtype == torch.uint8 else t.view({2: torch.int16, 4: torch.int32}[t.element_size()])


def run(state):
    kind = state["kind"]
    if kind == "sdpa":
        return state["op"].scaled_dot_product_attention(state["query"], state["key"], state["value"], None, state["input_pos"], state["positions"],
                                                        return_attn_weights=state["weights"], output_transposed=True, quant=state["quant"])
    if kind == "quantize":
        qz, (start, end) = state["quantizer"], state["range"]
        qz.quantize(start, end, state["rows"])
        return {"codes": qz.quant_buffer, "scale": _bits(qz.quant_scales), "zp": qz.quant_zero_points, "rows": _bits(qz.dequantize(start, end))}
    if kind == "model":
        return state["model"].prefill(state["ids"])
    cache = state["cache"]
    if kind == "prompt":
        cache.reset()
    out = cache.forward(*state["tokens"])
    got = {"out": out, "k": _bits(cache.k), "v": _bits(cache.v), "positions": cache.token_pos, "scores": cache.scores, "v_norm": cache.v_norm,
           "q_errors": cache.q_errors}
    if cache.quantized:
        got.update({n: _bits(getattr(cache, n)) for n in ("k_scale", "k_zp", "v_scale", "v_zp")})
    return got


# -- what a pass cannot do without ------------------------------------------------------------------------------


def _row_bytes(c):
    """Bytes of one K or V row of the store, with its scale and zero point."""
    bits = BITS[c["store"]]
    return c["D"] * bits // 8 + (0 if bits == 16 else 8)


def work(case):
    c, kind = case, case["kind"]
    if kind == "quantize":
        rows = c["B"] * c["Hkv"] * (c["end"] - c["start"])
        states = rows // c["Hkv"] if c["over_heads"] else rows
        codes = rows * c["D"] * c["bits"] // 8 + 8 * states
        return {"bytes": 2 * (2 * rows * c["D"] + codes), "flops": 0}
    if kind == "model":
        m = QWEN3_4B
        per_token = 2 * (m.n_embd * (m.n_head + 2 * m.n_query_groups) * m.head_size + m.n_head * m.head_size * m.n_embd + 3 * m.n_embd * m.intermediate_size)
        first, rest = c["T"], c["tokens"] - c["T"]
        attention = 4 * m.n_head * m.head_size * (first * first / 2 + rest * c["T"])
        weights = per_token  # two bytes a weight, two operations a weight and token
        chunks = 1 + -(-rest // c["chunk"])
        return {"bytes": c["layers"] * (weights * chunks + 4 * m.n_embd * c["tokens"]), "flops": c["layers"] * (per_token * c["tokens"] + attention)}
    B, Hq, Hkv, D, q, T = c["B"], c["Hq"], c["Hkv"], c["D"], c["q"], c["T"]
    in_out = 4 * B * Hq * q * D  # queries in, outputs out
    store = 2 * B * Hkv * T * _row_bytes(c)
    if kind == "sdpa":
        extra = 4 * B * Hkv * T * ((1 if c["weights"] else 0) + (1 if c["scattered"] and q > 1 else 0))
        return {"bytes": in_out + store + extra, "flops": 4 * B * Hq * q * T * D}
    new_rows = 2 * B * Hkv * q * (2 * D + _row_bytes(c))
    if kind == "prompt":
        return {"bytes": in_out + new_rows, "flops": 2 * B * Hq * q * q * D}
    slots = 4 * B * Hkv * T
    read = slots * (2 + (1 if q > 1 or c["normalize"] else 0) + (1 if "vlen" in c["policy"] else 0) + (1 if "qh2o" in c["policy"] else 0))
    return {"bytes": in_out + store + new_rows + read + 4 * B * Hkv * q, "flops": 4 * B * Hq * q * T * D}


def tolerance(case):
    if case["kind"] == "quantize":
        return "exact"  # codes, scales, zero points and dequantised rows are defined to the bit
    if case["kind"] == "model":
        return {"rel": 2e-2}  # bf16 activations through the layers, and slots whose scores tie to rounding
    # bf16 / fp16 outputs; the order of slots whose scores agree to rounding may change
    return {"rel": 1e-2, "differ": 1e-2}
