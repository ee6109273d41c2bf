"""The norms, the row activation and the row argmax where their launches
change: one, two or more vectors per lane, a last vector past the row, slice
groups of 2, 4 and 8, rows that end inside a workgroup of the activation,
and the target in any wavefront of the argmax (triton_ops.py:36-97, 106-122;
scheduler/continuous.py:265-275)."""

from __future__ import annotations

import pytest
import torch

from tensorforge_amd.kernels import argmax_rows, residual_rms_norm, rms_norm, swiglu_gate_up
from tensorforge_amd.kernels.ops import residual_rms_norm_partials

pytestmark = pytest.mark.gpu
# Half an ulp of the rounded result, relative.
HALF_ULP = {torch.float32: 2.0 ** -24, torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}


def _norm_bound(want, columns, dtype):
    # The fp32 sum of squares (half of its relative error reaches the scale),
    # rsqrtf, two products and one rounding; a subnormal step in fp16.
    return (HALF_ULP[dtype] + (columns / 2 + 8) * 2.0 ** -24) * want.abs() + 2.0 ** -24


@pytest.mark.parametrize("columns", [1, 8, 504, 512, 1016, 1032, 2048, 8184, 8192, 8200, 16384, 33, 1025])
@pytest.mark.parametrize("dtype", list(HALF_ULP))
def test_norm_vectors_per_lane(device, dtype, columns):
    generator = torch.Generator().manual_seed(columns)
    draw = lambda *shape: torch.randn(*shape, generator=generator).to(dtype).to(device)  # noqa: E731
    x, r, w = draw(5, columns), draw(5, columns), 1 + 0.1 * draw(columns)
    for residual in (None, r):
        total = x.double() if residual is None else x.double() + residual.double()
        want = total * torch.rsqrt(total.pow(2).mean(1, keepdim=True) + 1e-5) * w.double()
        if residual is None:
            norm = rms_norm(x, w, 1e-5)
        else:
            stored, norm = residual_rms_norm(x, residual, w, 1e-5)
            assert torch.equal(stored, (x.float() + residual.float()).to(dtype))
            in_place = residual.clone()  # the residual stream updated where it is
            again = residual_rms_norm(x, in_place, w, 1e-5, residual_output=in_place)[1]
            assert torch.equal(in_place, stored) and torch.equal(again, norm)
        assert ((norm.double() - want).abs() <= _norm_bound(want, columns, dtype)).all()


@pytest.mark.parametrize("columns", [8, 1024, 333])
def test_a_row_has_the_same_bits_in_calls_of_many_rows(device, columns):
    generator = torch.Generator().manual_seed(columns)
    x, r = (torch.randn(2049, columns, generator=generator).bfloat16().to(device) for _ in range(2))
    w = torch.rand(columns, generator=generator).bfloat16().to(device)
    many = residual_rms_norm(x, r, w, 1e-5)
    few = residual_rms_norm(x[-2048:], r[-2048:], w, 1e-5)
    assert torch.equal(many[0][-2048:], few[0]) and torch.equal(many[1][-2048:], few[1])


@pytest.mark.parametrize("splits", [1, 2, 3, 4, 5, 8, 9, 17])
@pytest.mark.parametrize("columns", [512, 2048, 2056, 4104, 99])
def test_slice_groups_add_in_slice_order(device, columns, splits):
    generator = torch.Generator().manual_seed(splits)
    partials = torch.randn(splits, 3, columns, generator=generator).to(device)
    r = torch.randn(3, columns, generator=generator).bfloat16().to(device)
    w = torch.rand(columns, generator=generator).bfloat16().to(device)
    running = partials[0].clone()
    for s in range(1, splits):
        running += partials[s]
    want = residual_rms_norm(running.bfloat16(), r, w, 1e-5)
    got = residual_rms_norm_partials(partials, r, w, 1e-5)
    assert torch.equal(got[0], want[0])
    # The two launches may take other workgroup sizes: sums in another order.
    assert ((got[1].double() - want[1].double()).abs()
            <= 2 * _norm_bound(want[1].double(), columns, torch.bfloat16)).all()


@pytest.mark.parametrize("rows,columns", [(1, 1), (1, 8), (3, 104), (1, 2048), (1, 2056), (1, 4096), (7, 5632), (65, 333)])
@pytest.mark.parametrize("dtype", list(HALF_ULP))
def test_activation_rows(device, dtype, rows, columns):
    generator = torch.Generator().manual_seed(rows + columns)
    wide = (2 * torch.randn(rows, 2 * columns + 8, generator=generator)).to(dtype).to(device)
    for gate_up in (wide[:, :2 * columns], wide[:, :2 * columns].contiguous(), wide[:, 3:3 + 2 * columns]):
        gate, up = gate_up[:, :columns].double(), gate_up[:, columns:].double()
        want = gate * torch.sigmoid(gate) * up
        backing = torch.full((rows, columns + 8), 7.0, dtype=dtype, device=device)
        got = swiglu_gate_up(gate_up, output=backing[:, :columns])
        # exp, the sum, the quotient and the product in fp32, and one rounding.
        bound = (HALF_ULP[dtype] + 16 * 2.0 ** -24) * want.abs() + 2.0 ** -24
        assert ((got.double() - want).abs() <= bound).all()
        assert (backing[:, columns:] == 7.0).all()  # nothing past a row's end


@pytest.mark.parametrize("columns", [1, 63, 8192, 32000, 40001])
@pytest.mark.parametrize("dtype", list(HALF_ULP))
def test_argmax_target_anywhere(device, dtype, columns):
    generator = torch.Generator().manual_seed(columns)
    logits = torch.randn(8, columns, generator=generator).clamp(-3, 3).to(dtype)
    places = sorted({0, columns - 1, columns // 2, columns // 3})
    for row, place in enumerate(places):
        logits[row, place] = 5
        logits[row, columns - 1] = 5  # a later tie loses
    logits[4] = -float("inf")
    logits[5, columns // 2] = float("nan")
    logits[5, columns - 1] = float("nan")
    logits[6] = 0.0
    logits[6, columns // 2] = -0.0
    logits[7, columns // 3] = float("inf")
    want = [int((row.isnan() if row.isnan().any() else row == row.max()).nonzero()[0]) for row in logits]
    assert argmax_rows(logits.to(device)).tolist() == want
