"""linear_kstream and the K-split SwiGLU at the edges of their tiles: last
chunks of 32, fewer chunks than wavefronts or ring buffers, ragged rows and
columns, padded row strides, and the same bits for a row whatever tile its
call takes (model/layers.py:88-95, 144-158)."""

from __future__ import annotations

import pytest
import torch

from tensorforge_amd.kernels import linear_kstream, linear_swiglu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [32, 64, 96, 160, 288, 1312, 2048])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_kstream_tile_edges(device, dtype, k):
    generator = torch.Generator().manual_seed(k)
    ulp = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)  # half an ulp, relative
    for n in (1, 23, 48, 333, 2600):
        x_all = torch.randn(64, k + 8, generator=generator).to(dtype).to(device)[:, :k]
        w = (torch.randn(n, k + 16, generator=generator) / k ** 0.5).to(dtype).to(device)[:, :k]
        wide = linear_kstream(x_all, w)
        for rows in (1, 15, 17, 33, 48, 49, 64):
            x = x_all[:rows]
            got = linear_kstream(x, w)
            want = x.double() @ w.double().T
            # fp32 sums of k products, then one rounding (and a subnormal step in fp16).
            bound = (k + 8) * 2.0 ** -23 * (x.double().abs() @ w.double().abs().T) + ulp * want.abs() + 2.0 ** -24
            assert ((got.double() - want).abs() <= bound).all(), (n, rows)
            assert torch.equal(got, wide[:rows]), (n, rows)  # no tile changes a row's bits
            normed = linear_kstream(x, w, norm_eps=1e-5)
            inv = torch.rsqrt(x.double().pow(2).mean(1, keepdim=True) + 1e-5)
            # The sum of squares and rsqrtf add a few roundings of the scale.
            assert ((normed.double() - inv * want).abs()
                    <= inv * bound + (k + 16) * 2.0 ** -23 * (inv * want).abs() + ulp * (inv * want).abs()
                    + 2.0 ** -24).all(), (n, rows)


@pytest.mark.parametrize("inter", [8, 23, 24, 100, 1000])
@pytest.mark.parametrize("norm", [None, 1e-5])
def test_kswiglu_tiles_give_the_bits_of_the_projection(device, inter, norm):
    k = 352
    generator = torch.Generator().manual_seed(inter)
    x_all = torch.randn(64, k, generator=generator).half().to(device)
    w = (torch.randn(2 * inter, k, generator=generator) / k ** 0.5).half().to(device)
    wide = linear_swiglu(x_all, w, k_split=True, norm_eps=norm)
    product = linear_kstream(x_all, w, norm_eps=norm).float()
    gate, up = product[:, :inter], product[:, inter:]
    want = gate.double() * torch.sigmoid(gate.double()) * up.double()
    # The activation's fp32 steps (a few ulps) and one rounding to fp16.
    assert ((wide.double() - want).abs() <= (2.0 ** -11 + 2.0 ** -20) * want.abs() + 2.0 ** -24).all()
    for rows in (1, 16, 31, 47, 64):
        assert torch.equal(linear_swiglu(x_all[:rows], w, k_split=True, norm_eps=norm), wide[:rows]), rows
