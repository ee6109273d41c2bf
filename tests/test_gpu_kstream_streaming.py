"""linear_kstream and the K-split SwiGLU on both sides of the rule that streams
weights past the caches: the same bits from line-aligned weights, from rows or a
base off the 128-byte lines, and from one or several row blocks."""

from __future__ import annotations

import pytest
import torch

from tensorforge_amd.kernels import linear_kstream, linear_swiglu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize(("n", "k"), [(1536, 2048), (1472, 2048), (736, 4224), (1024, 3008)])
def test_streamed_and_cached_weights_give_the_same_bits(device, n, k):
    generator = torch.Generator().manual_seed(n + k)
    x_all = torch.randn(64, k, generator=generator).bfloat16().to(device)
    w = (torch.randn(n, k, generator=generator) / k ** 0.5).bfloat16().to(device)  # around 6 MB
    padded = torch.empty(n, k + 8, dtype=w.dtype, device=device)[:, :k].copy_(w)
    shifted = torch.empty(n * k + 8, dtype=w.dtype, device=device)[8:].view(n, k).copy_(w)
    assert padded.stride(0) * 2 % 128 and shifted.data_ptr() % 128
    wide = linear_kstream(x_all, w)
    want = x_all.double() @ w.double().T
    bound = (k + 8) * 2.0 ** -23 * (x_all.double().abs() @ w.double().abs().T) + 2.0 ** -8 * want.abs()
    assert ((wide.double() - want).abs() <= bound).all()
    normed = linear_kstream(x_all, w, norm_eps=1e-5)
    act = linear_swiglu(x_all, w, k_split=True)
    for rows in (1, 16, 17, 32, 33, 48, 49, 64):
        x = x_all[:rows]
        for weight in (w, padded, shifted):
            assert torch.equal(linear_kstream(x, weight), wide[:rows]), rows
            assert torch.equal(linear_kstream(x, weight, norm_eps=1e-5), normed[:rows]), rows
            assert torch.equal(linear_swiglu(x, weight, k_split=True), act[:rows]), rows
