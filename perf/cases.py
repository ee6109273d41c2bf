"""Performance cases of the batched decode path: what each measures, its inputs, its pass, the work it cannot do without
and the same outputs in 64 bits.

A case's ``kind`` names the part of the path:

  decode_step        one graph-captured decode step of the 22-layer TinyLlama-geometry model
  prefill            the packed prefill of one or several prompts through that model
  decode_layer       one decoder layer of a decode step, its five launches called one by one
  attention          one paged decode-attention call
  prefill_attention  one packed causal attention call
  append             RoPE and the paged K/V append of packed prompts
  pointwise          a prefill layer's residual RMSNorm and SwiGLU
  head               the final RMSNorm, the LM head and greedy sampling of a decode step

Prompt lengths are written out ("271" or "730,509,261"); context lengths of decode rows are drawn from the seed.  The
whole-model cases run in float16: through 22 layers bfloat16 roundings add up to 3% of the logits, which would hide a
wrong result; the layers' own cases run in both.
"""

from __future__ import annotations

import dataclasses
import math
import random

import torch
from torch import Tensor

from tensorforge_amd.cache import PagedKVCache, PagedKVCacheConfig
from tensorforge_amd.decode import BucketedDecodeExecutor, DecoderWeights, tinyllama_config
from tensorforge_amd.kernels import (
    PagedAttentionWorkspace,
    argmax_rows,
    fold_norm_gain,
    linear_kstream,
    linear_stream,
    linear_swiglu,
    paged_gqa_decode_attention,
    residual_rms_norm,
    rms_norm,
    rope_paged_kv_append,
    swiglu_gate_up,
)
from tensorforge_amd.kernels.attention import paged_gqa_decode_attention_rope_append
from tensorforge_amd.kernels.prefill import prefill_attention, prefill_tiles
from tensorforge_amd.workloads import decode_attention_bytes, decode_attention_flops, decode_step_bytes

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
DEVICE = "cuda"
PAGE = 16
EPS = 1e-5
# 19 prompts of one admission of the serving workload (lognormal, median 256, clipped to [16, 2048]).
ADMISSION = "262,218,421,279,98,331,733,553,145,93,158,263,39,215,95,142,1661,304,2048"


def listed() -> list[dict]:
    return [
        # The headline decode step: a full batch of ragged requests up to 2k tokens.
        {"name": "decode_step_b64", "kind": "decode_step", "rows": 64, "low": 128, "high": 2047, "dtype": "fp16"},
        # Serving at a moderate rate: a request arrives alone and waits for its first token.
        {"name": "prefill_one", "kind": "prefill", "prompts": "271", "dtype": "fp16"},
        # A few requests admitted together.
        {"name": "prefill_packed", "kind": "prefill", "prompts": "730,509,261", "dtype": "fp16"},
        # One layer at the narrow batches of moderate load, where latency and launches count.
        {"name": "decode_layer_b4", "kind": "decode_layer", "rows": 4, "low": 64, "high": 1000, "dtype": "fp16"},
        # The headline attention call: 64 ragged rows and 8 padded ones.
        {"name": "attention_b64", "kind": "attention", "rows": 64, "padded": 8, "low": 128, "high": 2048,
         "query_heads": 32, "kv_heads": 4, "head_dim": 64, "page": 16, "dtype": "bf16"},
        # Long contexts, few rows (Llama-3-8B geometry).
        {"name": "attention_long", "kind": "attention", "rows": 4, "padded": 0, "low": 8192, "high": 32768,
         "query_heads": 32, "kv_heads": 8, "head_dim": 128, "page": 16, "dtype": "bf16"},
        # Full precision, as a caller checks a model or serves an fp32 one.
        {"name": "attention_fp32", "kind": "attention", "rows": 32, "padded": 0, "low": 64, "high": 2048,
         "query_heads": 32, "kv_heads": 4, "head_dim": 64, "page": 16, "dtype": "fp32"},
        # One layer's attention over a whole admission of prompts.
        {"name": "prefill_attention_admission", "kind": "prefill_attention", "prompts": ADMISSION,
         "query_heads": 32, "kv_heads": 4, "head_dim": 64, "dtype": "bf16"},
        # Long prompts at the Llama-3 geometry.
        {"name": "prefill_attention_long", "kind": "prefill_attention", "prompts": "4096,2051,777",
         "query_heads": 32, "kv_heads": 8, "head_dim": 128, "dtype": "fp16"},
        # One layer's RoPE and page writes of the admission.
        {"name": "append_admission", "kind": "append", "prompts": ADMISSION, "dtype": "bf16"},
        # One layer's norm and activation over the admission.
        {"name": "pointwise_admission", "kind": "pointwise", "tokens": 8058, "hidden": 2048, "inter": 5632,
         "dtype": "bf16"},
        # The end of a decode step: the vocabulary projection of 32 lanes.
        {"name": "head_b32", "kind": "head", "rows": 32, "dtype": "bf16"},
    ]


def _log_uniform(rng: random.Random, low: int, high: int) -> int:
    return min(high, max(low, round(math.exp(rng.uniform(math.log(low), math.log(high + 1))))))


def _prompt_lengths(rng: random.Random, total: int, most: int, longest: int) -> str:
    """Up to ``most`` lognormal prompt lengths of at most ``longest`` tokens, ``total`` tokens at most."""

    lengths: list[int] = []
    for _ in range(rng.randint(1, most)):
        length = min(longest, max(16, round(rng.lognormvariate(math.log(256), 0.8))), total - sum(lengths))
        if length < 1:
            break
        lengths.append(length)
    return ",".join(map(str, lengths))


def draw(rng: random.Random) -> dict:
    kind = rng.choice(["decode_step", "prefill", "decode_layer", "attention", "attention", "prefill_attention",
                       "append", "pointwise", "head"])
    half = rng.choice(["bf16", "bf16", "fp16"])
    if kind == "decode_step":
        high = _log_uniform(rng, 64, 2047)
        return {"kind": kind, "rows": _log_uniform(rng, 1, 64), "low": max(1, high // 16), "high": high, "dtype": "fp16"}
    if kind == "prefill":
        return {"kind": kind, "prompts": _prompt_lengths(rng, 1500, 4, 1500), "dtype": "fp16"}
    if kind == "decode_layer":
        high = _log_uniform(rng, 32, 2000)
        return {"kind": kind, "rows": _log_uniform(rng, 1, 64), "low": max(1, high // 16), "high": high, "dtype": half}
    if kind == "attention":
        dtype = rng.choice(["bf16", "bf16", "fp16", "fp32"])
        query_heads, kv_heads, head_dim = rng.choice([(32, 4, 64), (32, 8, 128), (8, 2, 32)])
        rows = _log_uniform(rng, 1, 64)
        size = 4 if dtype == "fp32" else 2
        budget = (64 << 20) if dtype == "fp32" else (256 << 20)
        most = budget // (rows * kv_heads * head_dim * 2 * size)
        high = _log_uniform(rng, 64, max(65, min(8192 if dtype == "fp32" else 32768, most)))
        return {"kind": kind, "rows": rows, "padded": rng.choice([0, 0, 3]), "low": max(1, high // 16), "high": high,
                "query_heads": query_heads, "kv_heads": kv_heads, "head_dim": head_dim, "page": rng.choice([16, 16, 32]),
                "dtype": dtype}
    if kind == "prefill_attention":
        query_heads, kv_heads, head_dim = rng.choice([(32, 4, 64), (32, 8, 128), (8, 2, 32)])
        total = _log_uniform(rng, 64, 6900)
        return {"kind": kind, "prompts": _prompt_lengths(rng, total, 19, 4096), "query_heads": query_heads,
                "kv_heads": kv_heads, "head_dim": head_dim, "dtype": half}
    if kind == "append":
        return {"kind": kind, "prompts": _prompt_lengths(rng, _log_uniform(rng, 16, 8058), 19, 2048), "dtype": half}
    if kind == "pointwise":
        hidden, inter = rng.choice([(2048, 5632), (4096, 14336), (256, 768)])
        return {"kind": kind, "tokens": _log_uniform(rng, 16, 8058 if hidden <= 2048 else 3000), "hidden": hidden,
                "inter": inter, "dtype": rng.choice([half, "fp32"])}
    return {"kind": kind, "rows": _log_uniform(rng, 1, 64), "dtype": half}


# -- inputs -------------------------------------------------------------------------------------------------------------


def _generator(seed: int) -> torch.Generator:
    return torch.Generator(device=DEVICE).manual_seed(seed)


def _normal(generator: torch.Generator, *shape: int, dtype: torch.dtype, std: float = 1.0) -> Tensor:
    return (torch.randn(*shape, generator=generator, device=DEVICE) * std).to(dtype)


def _lengths(case: dict) -> list[int]:
    return [int(n) for n in case["prompts"].split(",")]


def _row_lengths(case: dict, seed: int) -> list[int]:
    """Context lengths of a decode call's rows: uniform, the longest one present."""

    rng = random.Random(seed)
    lengths = [rng.randint(case["low"], case["high"]) for _ in range(case["rows"])]
    lengths[rng.randrange(case["rows"])] = case["high"]
    return lengths


def _expected_tokens(case: dict) -> float:
    return case["high"] + (case["rows"] - 1) * (case["low"] + case["high"]) / 2


def _tables(lengths: list[int], page: int, width: int, rng: random.Random) -> tuple[Tensor, int]:
    """Block tables over a permuted pool of exactly the pages the rows need."""

    counts = [-(-n // page) for n in lengths]
    pool = max(sum(counts), 1)
    order = list(range(pool))
    rng.shuffle(order)
    tables = torch.full((len(lengths), width), -1, dtype=torch.int32)
    at = 0
    for row, count in enumerate(counts):
        tables[row, :count] = torch.tensor(order[at:at + count], dtype=torch.int32)
        at += count
    return tables, pool


def _layer_model(dtype: torch.dtype, seed: int, layers: int = 1) -> DecoderWeights:
    config = dataclasses.replace(tinyllama_config(), num_hidden_layers=layers)
    return DecoderWeights.random(config, seed=seed, dtype=dtype, device=DEVICE)


def _model_cache(config, dtype: torch.dtype, lengths: list[int], max_sequences: int, seed: int) -> PagedKVCache:
    pages = sum(-(-(n + 1) // PAGE) for n in lengths)
    order = list(range(pages))
    random.Random(seed).shuffle(order)
    return PagedKVCache(PagedKVCacheConfig(
        num_layers=config.num_hidden_layers, num_blocks=pages, block_size=PAGE,
        num_kv_heads=config.num_key_value_heads, head_dim=config.head_dim, max_sequences=max_sequences,
        max_sequence_length=2048, dtype=dtype, device=torch.device(DEVICE)), page_order=order)


def prepare(case: dict, seed: int) -> dict:
    return globals()["_prepare_" + case["kind"]](case, seed)


def _prepare_decode_step(case: dict, seed: int) -> dict:
    config, dtype = tinyllama_config(), DTYPES[case["dtype"]]
    weights = _layer_model(dtype, seed, config.num_hidden_layers)
    lengths = [n - 1 for n in _row_lengths(case, seed)]  # tokens in the cache before the step
    rows = next(b for b in (1, 2, 4, 8, 16, 32, 64) if b >= len(lengths))
    context = next(c for c in (512, 1024, 2048) if c >= case["high"])
    cache = _model_cache(config, dtype, lengths, rows, seed)
    generator = _generator(seed + 1)
    for layer in range(config.num_hidden_layers):
        cache.key_cache[layer].normal_(generator=generator)
        cache.value_cache[layer].normal_(generator=generator)
    ids = [f"r{i}" for i in range(len(lengths))]
    for request_id, length in zip(ids, lengths):
        cache.create_sequence(request_id)
        if length:
            reservation = cache.begin_append(request_id, length)
            cache.record_all_layers_written(reservation)
            cache.commit(reservation)
    rng = random.Random(seed + 2)
    tokens = {request_id: rng.randrange(config.vocab_size) for request_id in ids}
    executor = BucketedDecodeExecutor(weights, cache, batch_buckets=(rows,), context_buckets=(context,))
    reservations = {request_id: cache.begin_append(request_id, 1) for request_id in ids}
    state = {"weights": weights, "cache": cache, "bucket": executor.bucket(len(ids), case["high"]),
             "ids": ids, "reservations": reservations, "tokens": tokens, "lengths": lengths}
    _run_decode_step(state)  # captures the bucket's graph
    return state


def _prepare_prefill(case: dict, seed: int) -> dict:
    config, dtype = tinyllama_config(), DTYPES[case["dtype"]]
    lengths = _lengths(case)
    weights = _layer_model(dtype, seed, config.num_hidden_layers)
    cache = _model_cache(config, dtype, lengths, len(lengths), seed)
    executor = BucketedDecodeExecutor(weights, cache, batch_buckets=(1,), context_buckets=(2048,))
    rng = random.Random(seed + 2)
    prompts = {f"r{i}": tuple(rng.randrange(config.vocab_size) for _ in range(n)) for i, n in enumerate(lengths)}
    return {"weights": weights, "executor": executor, "prompts": prompts}


def _prepare_decode_layer(case: dict, seed: int) -> dict:
    dtype = DTYPES[case["dtype"]]
    model = _layer_model(dtype, seed)
    config, layer = model.config, model.layers[0]
    lengths = _row_lengths(case, seed)  # the new token included
    capacity = -(-case["high"] // PAGE) * PAGE
    tables, pool = _tables(lengths, PAGE, capacity // PAGE, random.Random(seed))
    generator = _generator(seed + 1)
    rows, heads, kv_heads, dim = len(lengths), config.num_attention_heads, config.num_key_value_heads, config.head_dim
    positions = torch.tensor([n - 1 for n in lengths])
    pages = torch.tensor([int(tables[row, (n - 1) // PAGE]) for row, n in enumerate(lengths)], dtype=torch.int32)
    return {
        "config": config, "layer": layer, "lengths": lengths,
        "qkv": fold_norm_gain(layer.qkv, layer.input_norm), "gate_up": fold_norm_gain(layer.gate_up, layer.post_norm),
        "cos": model.rope_cos, "sin": model.rope_sin,
        "hidden": _normal(generator, rows, config.hidden_size, dtype=dtype),
        "key_cache": _normal(generator, pool, PAGE, kv_heads, dim, dtype=dtype),
        "value_cache": _normal(generator, pool, PAGE, kv_heads, dim, dtype=dtype),
        "tables": tables.to(DEVICE), "contexts": torch.tensor(lengths, dtype=torch.int32, device=DEVICE),
        "positions": positions.to(DEVICE), "pages": pages.to(DEVICE),
        "offsets": (positions % PAGE).to(torch.int32).to(DEVICE),
        "active": torch.ones(rows, dtype=torch.int32, device=DEVICE), "capacity": capacity,
        "attention": torch.empty(rows, heads, dim, dtype=dtype, device=DEVICE),
        "workspace": PagedAttentionWorkspace.allocate(batch_capacity=rows, query_heads=heads, head_dim=dim,
                                                      max_context_length=2 * capacity, device=torch.device(DEVICE)),
    }


def _prepare_attention(case: dict, seed: int) -> dict:
    dtype = DTYPES[case["dtype"]]
    lengths = _row_lengths(case, seed) + [0] * case["padded"]
    page, heads, kv_heads, dim = case["page"], case["query_heads"], case["kv_heads"], case["head_dim"]
    width = -(-case["high"] // page)
    tables, pool = _tables(lengths, page, width, random.Random(seed))
    generator = _generator(seed + 1)
    query = _normal(generator, len(lengths), heads, dim, dtype=dtype)
    return {
        "query": query, "key_cache": _normal(generator, pool, page, kv_heads, dim, dtype=dtype),
        "value_cache": _normal(generator, pool, page, kv_heads, dim, dtype=dtype), "tables": tables.to(DEVICE),
        "contexts": torch.tensor(lengths, dtype=torch.int32, device=DEVICE), "lengths": lengths, "capacity": width * page,
        "output": torch.empty_like(query),
        "workspace": PagedAttentionWorkspace.allocate(batch_capacity=len(lengths), query_heads=heads, head_dim=dim,
                                                      max_context_length=width * page, device=torch.device(DEVICE)),
    }


def _prepare_prefill_attention(case: dict, seed: int) -> dict:
    dtype = DTYPES[case["dtype"]]
    lengths = _lengths(case)
    total, heads, kv_heads, dim = sum(lengths), case["query_heads"], case["kv_heads"], case["head_dim"]
    generator = _generator(seed)
    q = _normal(generator, total, heads * dim, dtype=dtype)
    k = _normal(generator, total, kv_heads * dim, dtype=dtype)
    qkv = _normal(generator, total, (heads + 2 * kv_heads) * dim, dtype=dtype)
    return {"q": q, "k": k, "v": qkv[:, (heads + kv_heads) * dim:], "tiles": torch.from_numpy(prefill_tiles(lengths)).to(DEVICE),
            "output": torch.empty_like(q), "heads": heads, "kv_heads": kv_heads, "scale": dim ** -0.5}


def _prepare_append(case: dict, seed: int) -> dict:
    dtype = DTYPES[case["dtype"]]
    lengths = _lengths(case)
    config = tinyllama_config()
    heads, kv_heads, dim = config.num_attention_heads, config.num_key_value_heads, config.head_dim
    tables, pool = _tables(lengths, PAGE, -(-max(lengths) // PAGE), random.Random(seed))
    positions = torch.cat([torch.arange(n) for n in lengths])
    rows = torch.cat([torch.full((n,), row) for row, n in enumerate(lengths)])
    generator = _generator(seed)
    total = sum(lengths)
    angles = torch.outer(torch.arange(config.max_position_embeddings, dtype=torch.float32),
                         1.0 / config.rope_theta ** (torch.arange(0, dim, 2, dtype=torch.float32) / dim))
    angles = torch.cat((angles, angles), dim=-1)
    return {
        "qkv": _normal(generator, total, (heads + 2 * kv_heads) * dim, dtype=dtype), "positions": positions.to(DEVICE),
        "cos": angles.cos().to(dtype).to(DEVICE), "sin": angles.sin().to(dtype).to(DEVICE),
        "key_cache": torch.zeros(pool, PAGE, kv_heads, dim, dtype=dtype, device=DEVICE),
        "value_cache": torch.zeros(pool, PAGE, kv_heads, dim, dtype=dtype, device=DEVICE),
        "pages": tables[rows, positions // PAGE].to(torch.int32).to(DEVICE),
        "offsets": (positions % PAGE).to(torch.int32).to(DEVICE),
        "active": torch.ones(total, dtype=torch.int32, device=DEVICE), "heads": heads,
        "query": torch.empty(total, heads, dim, dtype=dtype, device=DEVICE),
        "key": torch.empty(total, kv_heads, dim, dtype=dtype, device=DEVICE),
    }


def _prepare_pointwise(case: dict, seed: int) -> dict:
    dtype = DTYPES[case["dtype"]]
    generator = _generator(seed)
    tokens, hidden, inter = case["tokens"], case["hidden"], case["inter"]
    return {"inputs": _normal(generator, tokens, hidden, dtype=dtype), "residual": _normal(generator, tokens, hidden, dtype=dtype),
            "weight": 1 + _normal(generator, hidden, dtype=dtype, std=0.1), "gate_up": _normal(generator, tokens, 2 * inter, dtype=dtype),
            "residual_output": torch.empty(tokens, hidden, dtype=dtype, device=DEVICE),
            "norm_output": torch.empty(tokens, hidden, dtype=dtype, device=DEVICE),
            "activation": torch.empty(tokens, inter, dtype=dtype, device=DEVICE)}


def _prepare_head(case: dict, seed: int) -> dict:
    config = tinyllama_config()
    dtype = DTYPES[case["dtype"]]
    generator = _generator(seed)
    rows = case["rows"]
    return {"hidden": _normal(generator, rows, config.hidden_size, dtype=dtype),
            "weight": 1 + _normal(generator, config.hidden_size, dtype=dtype, std=0.1),
            "lm_head": _normal(generator, config.vocab_size, config.hidden_size, dtype=dtype, std=0.02),
            "norm": torch.empty(rows, config.hidden_size, dtype=dtype, device=DEVICE),
            "logits": torch.empty(rows, config.vocab_size, dtype=dtype, device=DEVICE),
            "tokens": torch.empty(rows, dtype=torch.int64, device=DEVICE)}


# -- one pass -----------------------------------------------------------------------------------------------------------


def run(state: dict):
    if "bucket" in state:
        return _run_decode_step(state)
    if "prompts" in state:
        return _run_prefill(state)
    if "layer" in state:
        return _run_decode_layer(state)
    if "tiles" in state:
        return prefill_attention(state["q"], state["k"], state["v"], state["tiles"], query_heads=state["heads"],
                                 kv_heads=state["kv_heads"], scale=state["scale"], output=state["output"])
    if "gate_up" in state:
        residual, norm = residual_rms_norm(state["inputs"], state["residual"], state["weight"], EPS,
                                           residual_output=state["residual_output"], norm_output=state["norm_output"])
        return {"residual": residual, "norm": norm, "activation": swiglu_gate_up(state["gate_up"], output=state["activation"])}
    if "lm_head" in state:
        rms_norm(state["hidden"], state["weight"], EPS, output=state["norm"])
        linear_stream(state["norm"], state["lm_head"], output=state["logits"])
        argmax_rows(state["logits"], output=state["tokens"])
        return {"norm": state["norm"], "logits": state["logits"]}
    if "qkv" in state:
        rope_paged_kv_append(state["qkv"], state["positions"], state["cos"], state["sin"], state["key_cache"],
                             state["value_cache"], state["pages"], state["offsets"], state["active"],
                             query_heads=state["heads"], query_output=state["query"], key_output=state["key"])
        return {name: state[name] for name in ("query", "key", "key_cache", "value_cache")}
    return paged_gqa_decode_attention(state["query"], state["key_cache"], state["value_cache"], state["tables"],
                                      state["contexts"], max_context_length=state["capacity"], output=state["output"],
                                      workspace=state["workspace"])


def _run_decode_step(state: dict) -> Tensor:
    """The step's controls staged and its graph replayed.  The reservations stay open, so a pass can be repeated."""

    state["bucket"].prepare(state["ids"], state["reservations"], tokens=state["tokens"])
    state["bucket"].execute()
    return state["bucket"].logits[:len(state["ids"])]


def _run_prefill(state: dict) -> dict:
    """Fresh requests, their prompts' prefill, and the requests given back (their pages are free for the next pass)."""

    executor, prompts = state["executor"], state["prompts"]
    for request_id in prompts:
        executor.create_request(request_id)
    result = executor.prefill_prompts(prompts)
    if result.errors:
        raise RuntimeError(f"prefill failed: {result.errors}")
    for request_id in prompts:
        executor.release_request(request_id)
    return result.logits


def _run_decode_layer(state: dict) -> dict:
    layer = state["layer"]
    qkv = linear_kstream(state["hidden"], state["qkv"], norm_eps=EPS)
    attention = paged_gqa_decode_attention_rope_append(
        qkv, state["positions"], state["cos"], state["sin"], state["key_cache"], state["value_cache"], state["pages"],
        state["offsets"], state["active"], state["tables"], state["contexts"],
        query_heads=state["config"].num_attention_heads, max_context_length=state["capacity"], output=state["attention"],
        workspace=state["workspace"])
    residual = linear_kstream(attention.view(attention.shape[0], -1), layer.o_proj, residual=state["hidden"])
    act = linear_swiglu(residual, state["gate_up"], k_split=True, norm_eps=EPS)
    return {"qkv": qkv, "attention": attention, "residual": residual, "activation": act,
            "output": linear_kstream(act, layer.down, residual=residual)}


# -- the work of a pass -------------------------------------------------------------------------------------------------


def _attention_work(case: dict, size: int) -> tuple[float, float]:
    """Bytes and operations of a decode-attention call at the expected lengths of its rows."""

    tokens = _expected_tokens(case)
    lengths = [round(tokens / case["rows"])] * case["rows"]
    return (decode_attention_bytes(lengths, case["query_heads"], case["kv_heads"], case["head_dim"], case["page"], size),
            decode_attention_flops(lengths, case["query_heads"], case["head_dim"]))


def work(case: dict) -> dict:
    kind = case["kind"]
    config = tinyllama_config()
    h, f, d = config.hidden_size, config.intermediate_size, config.head_dim
    heads, kv_heads, layers = config.num_attention_heads, config.num_key_value_heads, config.num_hidden_layers
    size = 4 if case.get("dtype") == "fp32" else 2
    layer_params = (heads + 2 * kv_heads) * d * h + h * heads * d + 3 * f * h
    if kind == "decode_step":
        tokens, rows = _expected_tokens(case), case["rows"]
        return {"bytes": decode_step_bytes(config, tokens, rows, 2)["total"],
                "flops": 2 * rows * (layers * layer_params + config.vocab_size * h) + layers * 4 * heads * d * tokens}
    if kind == "prefill":
        lengths = _lengths(case)
        total = sum(lengths)
        pairs = sum(n * (n + 1) // 2 for n in lengths)
        return {"bytes": 2 * (layers * (layer_params + 2 * h + total * 2 * kv_heads * d) + config.vocab_size * (h + len(lengths))
                              + total * h),
                "flops": 2 * total * layers * layer_params + 2 * len(lengths) * config.vocab_size * h
                + layers * 4 * heads * d * pairs}
    if kind == "decode_layer":
        tokens, rows = _expected_tokens(case), case["rows"]
        return {"bytes": 2 * (layer_params + tokens * 2 * kv_heads * d + rows * (3 * h + 2 * kv_heads * d)),
                "flops": 2 * rows * layer_params + 4 * heads * d * tokens}
    if kind == "attention":
        nbytes, flops = _attention_work(case, size)
        return {"bytes": nbytes, "flops": flops}
    if kind == "prefill_attention":
        lengths = _lengths(case)
        q, kv = case["query_heads"] * case["head_dim"], case["kv_heads"] * case["head_dim"]
        return {"bytes": sum(lengths) * 2 * (2 * q + 2 * kv),
                "flops": 4 * q * sum(n * (n + 1) // 2 for n in lengths)}
    if kind == "append":
        total = sum(_lengths(case))
        return {"bytes": total * 2 * ((heads + 2 * kv_heads) * d + heads * d + 3 * kv_heads * d) + total * 20,
                "flops": 3 * total * (heads + kv_heads) * d}
    if kind == "pointwise":
        tokens = case["tokens"]
        return {"bytes": size * (tokens * (4 * case["hidden"] + 3 * case["inter"]) + case["hidden"]),
                "flops": tokens * (5 * case["hidden"] + 6 * case["inter"])}
    rows = case["rows"]
    return {"bytes": 2 * (config.vocab_size * h + rows * (2 * h + config.vocab_size) + h),
            "flops": 2 * rows * config.vocab_size * h}


def tolerance(case: dict) -> dict:
    """About four times what the present code is off from 64 bits: 0.0023 for one bf16 kernel and 0.004 at the end of a
    bf16 layer, an eighth of that in fp16 (0.0005, and 0.004 through the whole fp16 model), 5e-7 in fp32."""

    if case["kind"] in ("decode_step", "prefill"):
        return {"rel": 0.016}
    if case["dtype"] == "fp32":
        return {"rel": 4e-6}
    rel = 0.016 if case["kind"] == "decode_layer" else 0.01
    return {"rel": rel if case["dtype"] == "bf16" else rel / 8}


# -- the same outputs in 64 bits ----------------------------------------------------------------------------------------


def exact(case: dict, seed: int):
    return globals()["_exact_" + case["kind"]](case, prepare(case, seed))


def _norm64(x: Tensor, weight: Tensor) -> Tensor:
    x = x.double()
    return x * torch.rsqrt(x.square().mean(dim=-1, keepdim=True) + EPS) * weight.double()


def _rope64(x: Tensor, cos: Tensor, sin: Tensor) -> Tensor:
    """x [tokens, heads, D] rotated with each token's table rows."""

    half = x.shape[-1] // 2
    turned = torch.cat((-x[..., half:], x[..., :half]), dim=-1)
    return x * cos.double()[:, None] + turned * sin.double()[:, None]


def _attend64(q: Tensor, k: Tensor, v: Tensor, scale: float, causal: bool) -> Tensor:
    """q [T, Hq, D] over k, v [L, Hkv, D] (causal: T == L); one query head at a time."""

    group = q.shape[1] // k.shape[1]
    out = torch.empty(q.shape, dtype=torch.float64, device=q.device)
    for head in range(q.shape[1]):
        keys = k[:, head // group].double().t().contiguous()
        scores = q[:, head].double().contiguous() @ keys * scale
        if causal:
            scores.masked_fill_(torch.ones_like(scores, dtype=torch.bool).triu_(1), -math.inf)
        out[:, head] = torch.softmax(scores, dim=-1) @ v[:, head // group].double().contiguous()
    return out


def _rows_of(cache: Tensor, table: Tensor, length: int) -> Tensor:
    pages = cache[table[: -(-length // cache.shape[1])].long()]
    return pages.reshape(-1, *cache.shape[2:])[:length]


def _swiglu64(gate_up: Tensor) -> Tensor:
    gate, up = gate_up.double().chunk(2, dim=-1)
    return gate * torch.sigmoid(gate) * up


def _exact_attention(case: dict, state: dict) -> Tensor:
    out = torch.zeros(state["query"].shape, dtype=torch.float64, device=DEVICE)
    for row, length in enumerate(state["lengths"]):
        if length:
            out[row] = _attend64(state["query"][row:row + 1], _rows_of(state["key_cache"], state["tables"][row], length),
                                 _rows_of(state["value_cache"], state["tables"][row], length), case["head_dim"] ** -0.5, False)[0]
    return out


def _exact_prefill_attention(case: dict, state: dict) -> Tensor:
    dim = case["head_dim"]
    q, k, v = (t.reshape(t.shape[0], -1, dim) for t in (state["q"], state["k"], state["v"]))
    parts, at = [], 0
    for n in _lengths(case):
        parts.append(_attend64(q[at:at + n], k[at:at + n], v[at:at + n], state["scale"], True))
        at += n
    return torch.cat(parts).reshape(state["q"].shape)


def _exact_append(case: dict, state: dict) -> dict:
    heads, (kv_heads, dim) = state["heads"], state["key_cache"].shape[2:]
    x = state["qkv"].double().view(-1, heads + 2 * kv_heads, dim)
    cos, sin = state["cos"][state["positions"]], state["sin"][state["positions"]]
    q, k, v = _rope64(x[:, :heads], cos, sin), _rope64(x[:, heads:heads + kv_heads], cos, sin), x[:, heads + kv_heads:]
    key_cache, value_cache = state["key_cache"].double(), state["value_cache"].double()
    key_cache[state["pages"].long(), state["offsets"].long()] = k
    value_cache[state["pages"].long(), state["offsets"].long()] = v
    return {"query": q, "key": k, "key_cache": key_cache, "value_cache": value_cache}


def _exact_pointwise(case: dict, state: dict) -> dict:
    total = state["inputs"].double() + state["residual"].double()
    return {"residual": total, "norm": _norm64(total, state["weight"]), "activation": _swiglu64(state["gate_up"])}


def _exact_head(case: dict, state: dict) -> dict:
    norm = _norm64(state["hidden"], state["weight"])
    return {"norm": norm, "logits": norm @ state["lm_head"].double().t().contiguous()}


def _exact_decode_layer(case: dict, state: dict) -> dict:
    layer, config = state["layer"], state["config"]
    heads, kv_heads, dim = config.num_attention_heads, config.num_key_value_heads, config.head_dim
    hidden = state["hidden"].double()
    qkv = _norm64(hidden, layer.input_norm) @ layer.qkv.double().t().contiguous()
    x = qkv.view(-1, heads + 2 * kv_heads, dim)
    cos, sin = state["cos"][state["positions"]], state["sin"][state["positions"]]
    q, k, v = _rope64(x[:, :heads], cos, sin), _rope64(x[:, heads:heads + kv_heads], cos, sin), x[:, heads + kv_heads:]
    attention = torch.empty_like(q)
    for row, length in enumerate(state["lengths"]):
        keys = _rows_of(state["key_cache"], state["tables"][row], length).double()
        values = _rows_of(state["value_cache"], state["tables"][row], length).double()
        keys[-1], values[-1] = k[row], v[row]
        attention[row] = _attend64(q[row:row + 1], keys, values, dim ** -0.5, False)[0]
    residual = hidden + attention.reshape(hidden.shape) @ layer.o_proj.double().t().contiguous()
    act = _swiglu64(_norm64(residual, layer.post_norm) @ layer.gate_up.double().t().contiguous())
    return {"qkv": qkv, "attention": attention, "residual": residual, "activation": act,
            "output": residual + act @ layer.down.double().t().contiguous()}


def _exact_model(weights: DecoderWeights, tokens: Tensor, positions: Tensor, attend) -> Tensor:
    """The decoder over token rows; ``attend(layer, q, k, v)`` is each layer's attention over them.  Returns the last hidden
    rows after the final norm."""

    config = weights.config
    heads, kv_heads, dim = config.num_attention_heads, config.num_key_value_heads, config.head_dim
    residual = weights.embedding[tokens].double()
    cos, sin = weights.rope_cos[positions], weights.rope_sin[positions]
    for index, layer in enumerate(weights.layers):
        x = (_norm64(residual, layer.input_norm) @ layer.qkv.double().t().contiguous()).view(-1, heads + 2 * kv_heads, dim)
        q, k = _rope64(x[:, :heads], cos, sin), _rope64(x[:, heads:heads + kv_heads], cos, sin)
        attention = attend(index, q, k, x[:, heads + kv_heads:])
        residual = residual + attention.reshape(residual.shape) @ layer.o_proj.double().t().contiguous()
        act = _swiglu64(_norm64(residual, layer.post_norm) @ layer.gate_up.double().t().contiguous())
        residual = residual + act @ layer.down.double().t().contiguous()
    return _norm64(residual, weights.final_norm)


def _exact_decode_step(case: dict, state: dict) -> Tensor:
    weights, cache, ids = state["weights"], state["cache"], state["ids"]
    scale = weights.config.head_dim ** -0.5
    pages = [torch.tensor(cache.page_list(request_id)[0], device=DEVICE) for request_id in ids]

    def attend(layer: int, q: Tensor, k: Tensor, v: Tensor) -> Tensor:
        out = torch.empty_like(q)
        for row, length in enumerate(state["lengths"]):
            keys = torch.cat((_rows_of(cache.key_cache[layer], pages[row], length).double(), k[row:row + 1]))
            values = torch.cat((_rows_of(cache.value_cache[layer], pages[row], length).double(), v[row:row + 1]))
            out[row] = _attend_row64(q[row], keys, values, scale)
        return out

    tokens = torch.tensor([state["tokens"][request_id] for request_id in ids], device=DEVICE)
    hidden = _exact_model(weights, tokens, torch.tensor(state["lengths"], device=DEVICE), attend)
    return hidden @ weights.lm_head.double().t().contiguous()


def _attend_row64(q: Tensor, k: Tensor, v: Tensor, scale: float) -> Tensor:
    """One token's q [Hq, D] over k, v [L, Hkv, D], all heads together."""

    kv_heads = k.shape[1]
    grouped = q.view(kv_heads, -1, q.shape[-1])
    scores = torch.matmul(grouped, k.permute(1, 2, 0).contiguous()) * scale
    return torch.matmul(torch.softmax(scores, dim=-1), v.transpose(0, 1).contiguous()).reshape(q.shape)


def _exact_prefill(case: dict, state: dict) -> dict:
    weights = state["weights"]
    logits = {}
    for request_id, prompt in state["prompts"].items():
        positions = torch.arange(len(prompt), device=DEVICE)
        hidden = _exact_model(weights, torch.tensor(prompt, device=DEVICE), positions,
                              lambda _, q, k, v: _attend64(q, k, v, weights.config.head_dim ** -0.5, True))
        logits[request_id] = weights.lm_head.double() @ hidden[-1]
    return logits
