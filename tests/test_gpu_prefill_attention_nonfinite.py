"""Prefill attention around values that are not finite, against an fp64
restatement: they stay out of the queries whose key steps end before them, and
a query without any finite score answers NaN, not a number."""

from __future__ import annotations

import pytest
import torch

from tensorforge_amd.kernels.prefill import prefill_attention, prefill_tiles

pytestmark = pytest.mark.gpu

STEP = 32  # keys whose weights meet V together


def _run(device, q, k, v, lengths, hq, hkv, scale, heads_per_wave):
    out = torch.empty_like(q, device=device)
    prefill_attention(q.to(device), k.to(device), v.to(device),
                      torch.from_numpy(prefill_tiles(lengths)).to(device), query_heads=hq,
                      kv_heads=hkv, scale=scale, output=out, heads_per_wave=heads_per_wave)
    return out.cpu()


def _inputs(hq, hkv, d, dtype, total):
    generator = torch.Generator().manual_seed(total + d)
    return tuple(torch.randn(total, h * d, generator=generator).to(dtype) for h in (hq, hkv, hkv))


@pytest.mark.parametrize(("hq", "hkv", "d", "dtype"), [
    (8, 2, 64, torch.float16), (8, 2, 32, torch.bfloat16), (4, 1, 128, torch.float16)])
@pytest.mark.parametrize("heads_per_wave", [1, 4])
@pytest.mark.parametrize("bad", [16, 33, 47, 63, 96])
def test_a_value_that_is_not_finite_stays_out_of_earlier_steps(device, hq, hkv, d, dtype, heads_per_wave,
                                                               bad):
    lengths = [7, 131]
    q, k, v = _inputs(hq, hkv, d, dtype, sum(lengths))
    clean = _run(device, q, k, v, lengths, hq, hkv, d ** -0.5, heads_per_wave)
    v[lengths[0] + bad] = float("inf")
    out = _run(device, q, k, v, lengths, hq, hkv, d ** -0.5, heads_per_wave)
    # A wavefront's 16 queries take whole steps up to the one its last query ends in.
    tile_end = (torch.arange(lengths[1]) // 16 + 1) * 16
    before = (tile_end + STEP - 1) // STEP * STEP <= bad // STEP * STEP
    keep = torch.cat((torch.ones(lengths[0], dtype=torch.bool), before))
    assert torch.equal(out[keep], clean[keep])
    assert not torch.isfinite(out[lengths[0] + bad:]).any()


@pytest.mark.parametrize(("hq", "hkv", "d", "dtype"), [
    (8, 2, 64, torch.float16), (8, 2, 32, torch.bfloat16), (4, 1, 128, torch.bfloat16)])
@pytest.mark.parametrize(("score", "keys"), [(-float("inf"), 1), (-float("inf"), 70), (float("inf"), 1)])
def test_scores_that_are_not_finite(device, hq, hkv, d, dtype, score, keys):
    lengths = [1, 100]
    q, k, v = _inputs(hq, hkv, d, dtype, sum(lengths))
    q[:, ::d] = 1.0  # dimension 0 of every head meets the infinite key elements
    start = lengths[0]
    k[0, ::d] = score
    k[start:start + keys, ::d] = score
    out = _run(device, q, k, v, lengths, hq, hkv, d ** -0.5, 0).double()
    # A softmax over infinities: NaN from the first +inf on, and where -inf is all there is.
    nan = torch.ones(sum(lengths), dtype=torch.bool)
    if score < 0:
        nan[start + keys:] = False
    assert torch.isnan(out[nan]).all() and torch.isfinite(out[~nan]).all()
    if score < 0:  # -inf keys weigh nothing: as if the prompt began after them
        qs, ks, vs = (t[start + keys:].double().view(-1, h, d) for t, h in ((q, hq), (k, hkv), (v, hkv)))
        n = qs.shape[0]
        mask = torch.triu(torch.ones(n, n, dtype=torch.bool), 1)
        # Rounded weights against an unrounded sum (two ulp / 2), then the output's own rounding.
        eps = torch.finfo(dtype).eps / 2
        for h in range(hq):
            scores = (qs[:, h] @ ks[:, h // (hq // hkv)].T * d ** -0.5).masked_fill(mask, -float("inf"))
            weights = torch.softmax(scores, dim=-1)
            values = vs[:, h // (hq // hkv)]
            want, size = weights @ values, weights @ values.abs()
            got = out[start + keys:].view(n, hq, d)[:, h]
            assert bool(((got - want).abs() <= 3 * eps * size + eps * want.abs() + 1e-6).all())
