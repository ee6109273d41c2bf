"""Which weights a prefill takes: an embedding table with padded rows, and none
that gradients are to reach (the kernels are inference-only)."""

from __future__ import annotations

import dataclasses

import pytest
import torch

from tensorforge_amd.cache import PagedKVCache, PagedKVCacheConfig
from tensorforge_amd.decode import DecoderWeights, prefill_requests, small_config

pytestmark = pytest.mark.gpu

PROMPTS = {"a": list(range(1, 18)), "b": [7] * 70}


def _model(device):
    config = small_config()
    cache = PagedKVCache(PagedKVCacheConfig(
        num_layers=config.num_hidden_layers, num_blocks=16, block_size=16,
        num_kv_heads=config.num_key_value_heads, head_dim=config.head_dim, max_sequences=2,
        max_sequence_length=128, dtype=torch.float16, device=device))
    return DecoderWeights.random(config, seed=2, dtype=torch.float16, device=device), cache


def _prefill(weights, cache):
    for request_id in PROMPTS:
        cache.create_sequence(request_id)
    result = prefill_requests(weights, cache, PROMPTS)
    for request_id in PROMPTS:
        cache.release(request_id)
    return result


def test_prefill_takes_an_embedding_of_padded_rows(device):
    weights, cache = _model(device)
    want = _prefill(weights, cache)
    vocab, hidden = weights.embedding.shape
    padded = torch.empty(vocab, hidden + 8, dtype=torch.float16, device=device)[:, :hidden].copy_(weights.embedding)
    got = _prefill(dataclasses.replace(weights, embedding=padded), cache)
    assert not want.errors and not got.errors
    assert all(torch.equal(got.logits[request_id], want.logits[request_id]) for request_id in PROMPTS)


@pytest.mark.parametrize("name", ["o_proj", "down"])
def test_prefill_refuses_weights_that_require_grad(device, name):
    weights, cache = _model(device)
    want = _prefill(weights, cache)
    getattr(weights.layers[1], name).requires_grad_(True)
    result = _prefill(weights, cache)
    assert not result.logits and all("inference-only" in message for message in result.errors.values())
    with torch.no_grad():
        result = _prefill(weights, cache)
    assert not result.errors
    assert all(torch.equal(result.logits[request_id], want.logits[request_id]) for request_id in PROMPTS)
