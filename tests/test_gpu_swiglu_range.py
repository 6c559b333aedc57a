"""The bf16 GEMM + SwiGLU at widths of no whole tile (a width that is no multiple of 128, a reduction that
is no multiple of 64) over gates and ups whose product, or whose exp(-gate), leaves the f32 range while the
result does not, for groups of few rows and of many.

One product per sum, so the gate and up values are exact: the result is silu(gate) * up rounded once
(2^-9 of a value), with a few f32 roundings before: 2^-8 bounds both.
"""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

PAIRS = [(-1e20, 1e20), (-2.0, 3e38), (-88.5, 1e30), (3.0, 1.0), (-20.0, 2.0), (100.0, -2.5), (1e20, 1e10), (-60.0, 1e20)]


@pytest.mark.parametrize("rows", [3, 70])
@pytest.mark.parametrize("Kin,I", [(64, 72), (40, 128), (200, 264)])
def test_swiglu_keeps_its_range(dev, rows, Kin, I):
    from mintext_amd.kernels.grouped_matmul import grouped_matmul_swiglu

    E = 2
    g, u = (torch.tensor([p[i] for p in PAIRS] * (I // 8), device=dev).bfloat16() for i in (0, 1))
    x = torch.zeros(rows * E, Kin, device=dev, dtype=torch.bfloat16)
    x[:, Kin - 1] = 1.0
    w = torch.zeros(E, Kin, 2 * I, device=dev, dtype=torch.bfloat16)
    w[:, Kin - 1, :I] = g
    w[:, Kin - 1, I:] = u
    y = grouped_matmul_swiglu(x, w, torch.full((E,), rows, dtype=torch.int32, device=dev)).double()
    want = torch.nn.functional.silu(g.double()) * u.double()
    assert ((y - want).abs() <= 2.0 ** -8 * want.abs()).all()
