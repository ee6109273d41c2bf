"""Prefill attention where its 64-key chunks and lazily raised maxima can go
wrong: prompts around the chunk and block edges, enough workgroups for the
two-heads form and the die-wise head order, scores that keep rising or
falling along the prompt.

Bar, per element against an fp64 restatement with weights w: the weights are
rounded to the storage type (half an ulp u each), independent errors of at most
u w |v| whose sum passes 7 u sqrt(sum (w v)^2) with probability 2 exp(-24.5)
(Hoeffding), below one in a thousand over a case's elements; the fp32 scores,
exponentials and sums add their worst case; the output is rounded once.  A key
left out or counted twice, anywhere in the longest prompt, lies outside it."""

from __future__ import annotations

import pytest
import torch

from tensorforge_amd.kernels.prefill import prefill_attention, prefill_tiles

pytestmark = pytest.mark.gpu


U = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}
FP32 = 2.0 ** -24


def _reference(q, k, v, lengths, hq, hkv, d, scale, bias=None):
    """fp64 outputs and the bar; ``bias`` (for planted mistakes) is added to
    the scores of the last prompt's keys."""

    out = torch.zeros(q.shape[0], hq, d, dtype=torch.float64, device=q.device)
    bar = torch.zeros_like(out)
    u, start = U[q.dtype], 0
    tiny = 2.0 ** -25 if q.dtype == torch.float16 else 0.0  # half a subnormal step of a weight
    for prompt, n in enumerate(lengths):
        qs, ks, vs = (t[start:start + n].double().view(n, -1, d).transpose(0, 1).contiguous() for t in (q, k, v))
        mask = torch.triu(torch.ones(n, n, dtype=torch.bool, device=q.device), 1)
        for h in range(hq):
            kt, value = ks[h // (hq // hkv)].T.contiguous(), vs[h // (hq // hkv)]
            scores = qs[h] @ kt * scale
            if bias is not None and prompt == len(lengths) - 1:
                scores = scores + bias
            w = torch.softmax(scores.masked_fill(mask, -float("inf")), dim=-1)
            y, size = w @ value, w @ value.abs()
            # Relative error of a weight: the score's fp32 products and sums, its
            # scaling, the exponential; a sum over n of them with weights of 2^8.
            off = w * ((d + 8) * FP32 * (qs[h].abs() @ kt.abs()) * scale + 2.0 ** -21)
            rows = slice(start, start + n)
            out[rows, h] = y
            bar[rows, h] = (7 * u * torch.sqrt(w.square() @ value.square()) + off @ value.abs()
                            + off.sum(1, keepdim=True) * y.abs() + 2 * (n + 8) * FP32 * size
                            + u * y.abs() + tiny * value.abs().sum(0))
        start += n
    return out.view(q.shape[0], hq * d), bar.view(q.shape[0], hq * d)


@pytest.mark.parametrize(("hq", "hkv", "d", "dtype", "lengths", "growth", "scale"), [
    # 600 or more two-head workgroups; 16 head groups a block (a multiple of the dies).
    (32, 4, 64, torch.bfloat16, [63, 64, 65, 127, 128, 129, 191, 192, 193, 1, 500, 700], 0.0, 0.125),
    (32, 8, 128, torch.float16, [64, 65, 640, 129, 1, 63, 200, 33, 700], 0.0, 128 ** -0.5),
    # Scores that rise by far more than 2^8 along the prompt, and fall from a high start.
    (8, 2, 64, torch.float16, [130, 64, 257], 0.06, 0.125),
    (8, 2, 64, torch.float16, [130, 64, 257], -0.004, 0.6),
    (8, 2, 32, torch.bfloat16, [90, 200], 0.05, 0.2),
    (16, 4, 128, torch.bfloat16, [150, 70], 0.03, 0.1),
    (6, 6, 64, torch.bfloat16, [3, 65], 0.0, 1.0),
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
    q, k, v = q.to(device), k.to(device), v.to(device)
    want, bar = _reference(q, k, v, lengths, hq, hkv, d, scale)
    assert ((out.double() - want).abs() <= bar).all()
    if growth == 0 and scale < 1:  # every key of the last token has a weight near 1 / n
        n = lengths[-1]
        for key in (0, n // 2, n - 2):
            for change in (-float("inf"), 0.6931471805599453):  # left out; counted twice
                bias = torch.zeros(n, dtype=torch.float64, device=device)
                bias[key] = change
                wrong, _ = _reference(q, k, v, lengths, hq, hkv, d, scale, bias)
                assert ((out.double() - wrong)[-1].abs() > bar[-1]).any(), (key, change)
