"""The rule that chooses a form of the residual norm by the size of the call: a
row has the same bits on both sides of each line."""

from __future__ import annotations

import pytest
import torch

from tensorforge_amd.kernels import residual_rms_norm

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
