"""The prefill projections (tf_prefill_linear) against fp32 products, in
every output form and tile, at row, column and K counts around the tiles'
edges; and the one-call layer against the same launches made one by one.

Bars: the rounded product within one rounding (2^-8 bf16, 2^-11 fp16) of the
fp64 product plus 1e-5 of the row-by-column norm product (fp32 accumulation
over K <= 5632); slice sums within the second term alone."""

from __future__ import annotations

import random

import pytest
import torch
from torch.nn import functional as F

from tensorforge_amd import _native
from tensorforge_amd.cache import PagedKVCache, PagedKVCacheConfig
from tensorforge_amd.decode import (
    DecoderConfig,
    DecoderWeights,
    _NativePrefill,
    prefill_batch,
    tinyllama_config,
)
from tensorforge_amd.kernels.linear import linear_partials_sum, prefill_linear, prefill_linear_supported

pytestmark = pytest.mark.gpu

ROUNDING = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}
TILES = 10


def _operands(m, n, k, dtype, device, seed, x_pad=0, w_pad=0):
    generator = torch.Generator().manual_seed(seed)
    x = torch.randn(m, k + x_pad, generator=generator).to(dtype).to(device)[:, :k]
    w = (torch.randn(n, k + w_pad, generator=generator) * 0.05).to(dtype).to(device)[:, :k]
    return x, w


def _check(got, x, w, rounding, what):
    want = x.double() @ w.double().t().contiguous()
    bar = rounding * want.abs() + 1e-5 * x.double().norm(dim=1)[:, None] * w.double().norm(dim=1)[None]
    off = (got.double() - want).abs()
    assert bool((off <= bar).all()), f"{what}: off by {float((off - bar).max()):.3g} over the bar"


@pytest.mark.parametrize("tile", range(TILES + 1))
@pytest.mark.parametrize(("m", "n", "k", "splits", "x_pad", "w_pad"), [
    (1, 8, 256, 1, 0, 0), (65, 72, 256, 1, 8, 0), (129, 264, 320, 1, 0, 16), (257, 328, 512, 2, 8, 8),
    (97, 200, 1088, 4, 0, 0), (320, 64, 832, 3, 0, 0),
])
def test_prefill_linear_edges(device, tile, m, n, k, splits, x_pad, w_pad):
    dtype = torch.bfloat16 if (m + tile) % 2 else torch.float16
    x, w = _operands(m, n, k, dtype, device, seed=m + k, x_pad=x_pad, w_pad=w_pad)
    out = torch.full((m, n + 8), float("nan"), dtype=dtype, device=device)
    got = prefill_linear(x, w, output=out[:, :n], tile=tile)
    _check(got, x, w, ROUNDING[dtype], f"tile {tile}")
    assert bool(out[:, n:].isnan().all()), "columns past the output were written"
    if splits > 1:
        partials = torch.full((splits, m, n), float("nan"), device=device)
        prefill_linear(x, w, splits=splits, partials=partials, tile=tile)
        _check(partials.double().sum(0), x, w, 0.0, f"tile {tile}: slices")
        _check(linear_partials_sum(partials, dtype=dtype), x, w, ROUNDING[dtype], f"tile {tile}: summed")
    if n % 16 == 0:
        return
    act = prefill_linear(x, w, swiglu=True, tile=tile)
    product = F.linear(x.float(), w.float()).to(dtype).double()
    gate, up = product[:, :n // 2], product[:, n // 2:]
    want = gate * torch.sigmoid(gate) * up
    # The activation of products one rounding away from the reference's.
    bar = 6 * ROUNDING[dtype] * (want.abs() + gate.abs() * up.abs()) + 1e-4
    assert bool(((act.double() - want).abs() <= bar).all()), f"tile {tile}: swiglu"


@pytest.mark.parametrize("m", [65, 271, 1000, 2049])
def test_prefill_linear_chooses_slices_that_fill_its_tile(device, m):
    for n, k in ((2560, 2048), (2048, 5632), (1024, 256), (256, 768)):
        splits = _native.library().tf_prefill_linear_splits(m, n, k)
        assert 1 <= splits <= 4
        x, w = _operands(m, n, k, torch.float16, device, seed=k)
        partials = torch.empty(splits, m, n, device=device)
        prefill_linear(x, w, splits=splits, partials=partials)
        _check(partials.double().sum(0), x, w, 0.0, f"{m} x {n} x {k} in {splits}")


def test_prefill_linear_refuses_what_it_cannot_run(device):
    x, w = _operands(70, 64, 512, torch.float16, device, seed=0)
    assert not prefill_linear_supported(x[:, :200], w[:, :200])
    assert not prefill_linear_supported(x.float(), w.float())
    assert not prefill_linear_supported(x[:, 1:257], w[:, 1:257])  # rows off 16 bytes
    assert _native.library().tf_prefill_linear_splits(70, 64, 96) == 0
    with pytest.raises(RuntimeError, match="fill its load ring"):
        prefill_linear(x, w, splits=8, partials=torch.empty(8, 70, 64, device=device))


def _model(config: DecoderConfig, dtype, device, prompts):
    weights = DecoderWeights.random(config, seed=3, dtype=dtype, device=device)
    generator = torch.Generator(device=device).manual_seed(5)
    for layer in weights.layers:
        layer.input_norm.copy_(1 + 0.1 * torch.randn(config.hidden_size, generator=generator, device=device))
        layer.post_norm.copy_(1 + 0.1 * torch.randn(config.hidden_size, generator=generator, device=device))

    def fill() -> tuple[dict, PagedKVCache]:
        pages = sum(-(-len(p) // 16) for p in prompts.values())
        order = list(range(pages))
        random.Random(1).shuffle(order)
        cache = PagedKVCache(PagedKVCacheConfig(
            num_layers=config.num_hidden_layers, num_blocks=pages, block_size=16,
            num_kv_heads=config.num_key_value_heads, head_dim=config.head_dim, max_sequences=len(prompts),
            max_sequence_length=2048, dtype=dtype, device=device), page_order=order)
        cache.key_cache.zero_()
        cache.value_cache.zero_()
        for request_id in prompts:
            cache.create_sequence(request_id)
        return prefill_batch(weights, cache, prompts), cache

    return fill


@pytest.mark.parametrize(("layers", "dtype", "lengths"), [
    (2, torch.float16, [271]), (2, torch.bfloat16, [1, 65, 130]), (1, torch.float16, [1100, 700]),
    (2, torch.bfloat16, [16]),
])
def test_native_layers_match_the_launches_one_by_one(device, monkeypatch, layers, dtype, lengths):
    """TinyLlama layers through tf_prefill_layer and through the separate
    launches with library projections: the same first-layer pages up to the
    projections' sum order, and logits within the roundings of two layers."""

    import dataclasses

    config = dataclasses.replace(tinyllama_config(), num_hidden_layers=layers, vocab_size=512)
    rng = random.Random(7)
    prompts = {f"r{i}": [rng.randrange(512) for _ in range(n)] for i, n in enumerate(lengths)}
    fill = _model(config, dtype, device, prompts)
    got, got_cache = fill()
    monkeypatch.setattr(_NativePrefill, "supported", staticmethod(lambda *_: False))
    want, want_cache = fill()
    step = ROUNDING[dtype]
    for name in ("key_cache", "value_cache"):
        a, b = getattr(got_cache, name)[0].double(), getattr(want_cache, name)[0].double()
        # One rounding each of the projection (keys: and of the rotation).
        assert float((a - b).abs().max()) <= 4 * step * float(b.abs().max()), name
        assert float((a - b).norm()) <= step * float(b.norm()), name
    for request_id in prompts:
        a, b = got[request_id][1].double(), want[request_id][1].double()
        assert float((a - b).norm()) <= 8 * step * layers * float(b.norm()), request_id
