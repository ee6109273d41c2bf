"""Prefill attention where its 64-key chunks and lazily raised maxima can go
wrong: prompts around the chunk and block edges, enough workgroups for the
two-heads form and the die-wise head order, scores that keep rising or
falling along the prompt.  Bar: 2e-2 + 1e-2 |x|
against an fp64 restatement, the bar of the other prefill attention tests."""

from __future__ import annotations

import pytest
import torch

from helpers import NORTH_STAR_ATOL, NORTH_STAR_RTOL, assert_close
from tensorforge_amd.kernels.prefill import prefill_attention, prefill_tiles

pytestmark = pytest.mark.gpu


def _reference(q, k, v, lengths, hq, hkv, d, scale):
    out = torch.zeros(q.shape[0], hq, d, dtype=torch.float64)
    start = 0
    for n in lengths:
        qs, ks, vs = (t[start:start + n].double().view(n, -1, d) for t in (q, k, v))
        mask = torch.triu(torch.ones(n, n, dtype=torch.bool), 1)
        for h in range(hq):
            kv = h // (hq // hkv)
            scores = (qs[:, h] @ ks[:, kv].T * scale).masked_fill(mask, -float("inf"))
            out[start:start + n, h] = torch.softmax(scores, dim=-1) @ vs[:, kv]
        start += n
    return out.view(q.shape[0], hq * d)


@pytest.mark.parametrize(("hq", "hkv", "d", "dtype", "lengths", "growth", "scale"), [
    # 600 or more two-head workgroups; 16 head groups a block (a multiple of the dies).
    (32, 4, 64, torch.bfloat16, [63, 64, 65, 127, 128, 129, 191, 192, 193, 1, 500, 700], 0.0, 0.125),
    (32, 8, 128, torch.float16, [64, 65, 640, 129, 1, 700, 63, 200, 33], 0.0, 128 ** -0.5),
    # Scores that rise by far more than 2^8 along the prompt, and fall from a high start.
    (8, 2, 64, torch.float16, [130, 64, 257], 0.06, 0.125),
    (8, 2, 64, torch.float16, [130, 64, 257], -0.004, 0.6),
    (8, 2, 32, torch.bfloat16, [90, 200], 0.05, 0.2),
    (16, 4, 128, torch.bfloat16, [150, 70], 0.03, 0.1),
    (6, 6, 64, torch.bfloat16, [65, 3], 0.0, 1.0),
])
def test_prefill_attention_chunks(device, hq, hkv, d, dtype, lengths, growth, scale):
    total = sum(lengths)
    generator = torch.Generator().manual_seed(total)
    q = torch.randn(total, hq * d, generator=generator).to(dtype)
    k = torch.randn(total, hkv * d, generator=generator)
    position = torch.cat([torch.arange(n) for n in lengths])
    k = (k * (1 + growth * position)[:, None].clamp(min=0.05)).to(dtype)
    v = torch.randn(total, hkv * d, generator=generator).to(dtype)
    out = torch.full((total, hq * d), float("nan"), dtype=dtype, device=device)
    prefill_attention(q.to(device), k.to(device), v.to(device),
                      torch.from_numpy(prefill_tiles(lengths)).to(device), query_heads=hq,
                      kv_heads=hkv, scale=scale, output=out)
    assert_close(out.cpu(), _reference(q, k, v, lengths, hq, hkv, d, scale).float(), NORTH_STAR_ATOL,
                 NORTH_STAR_RTOL, f"hq={hq} hkv={hkv} d={d} growth={growth}")
