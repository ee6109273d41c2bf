"""The rules that choose a form of the residual norm and of RoPE by the size of
the call: a row has the same bits on both sides of each line."""

from __future__ import annotations

import pytest
import torch

from tensorforge_amd.kernels import residual_rms_norm, rope_paged_kv_append

pytestmark = pytest.mark.gpu

L1_BYTES = 8 << 20  # of one array, over all compute units: past it no loads run ahead


@pytest.mark.parametrize("columns", [1024, 2048, 4104, 8200, 12288, 16384])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_residual_norm_on_both_sides_of_the_l1s(device, dtype, columns):
    rows = -(-L1_BYTES // (columns * dtype.itemsize))  # the first size past the line
    generator = torch.Generator(device=device).manual_seed(columns)
    x, r = (torch.randn(rows, columns, generator=generator, device=device).to(dtype) for _ in range(2))
    w = torch.rand(columns, generator=generator, device=device).to(dtype)
    many = residual_rms_norm(x, r, w, 1e-5)
    few = residual_rms_norm(x[1:], r[1:], w, 1e-5)
    one = residual_rms_norm(x[-1:], r[-1:], w, 1e-5)
    for a, b, c in zip(many, few, one):
        assert torch.equal(a[1:], b) and torch.equal(a[-1:], c)
    assert torch.equal(many[0], (x.float() + r.float()).to(dtype))


@pytest.mark.parametrize(("heads", "kv_heads", "head_dim"), [(8, 2, 32), (4, 4, 64), (6, 2, 64), (30, 2, 16), (7, 1, 80)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_rope_on_both_sides_of_the_narrow_form(device, dtype, heads, kv_heads, head_dim):
    batch = 513  # one token past the narrow form's most; 256 pairs or just above a token
    generator = torch.Generator(device=device).manual_seed(head_dim)
    draw = lambda *shape: torch.randn(*shape, generator=generator, device=device).to(dtype)  # noqa: E731
    qkv, cos, sin = draw(batch, (heads + 2 * kv_heads) * head_dim), draw(600, head_dim), draw(600, head_dim)
    positions = torch.arange(batch, device=device)
    pages, offsets = (positions // 16).int(), (positions % 16).int()
    active = (positions % 5 != 3).int()

    def run(count):
        key_cache = torch.zeros(33, 16, kv_heads, head_dim, dtype=dtype, device=device)
        value_cache, key = torch.zeros_like(key_cache), torch.zeros(count, kv_heads, head_dim, dtype=dtype, device=device)
        query = rope_paged_kv_append(qkv[:count], positions[:count], cos, sin, key_cache, value_cache,
                                     pages[:count], offsets[:count], active[:count], query_heads=heads,
                                     key_output=key)
        return query, key, key_cache.flatten(0, 1)[:count], value_cache.flatten(0, 1)[:count]

    for wide, narrow in zip(run(batch), run(batch - 1)):
        assert torch.equal(wide[:batch - 1], narrow)
