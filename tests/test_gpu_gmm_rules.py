"""Which kernel of the grouped GEMM takes a call, on both sides of the rules that choose by size (each rule's
comment has the times of both kernels), and the parity of what was chosen.

Parity: against float64 on the same bf16 operands, at 2.5e-3 in the 2-norm (one rounding of 2^-9 a value,
and f32 sums below 2^-15 of the result).
"""
from __future__ import annotations

import numpy as np
import pytest
import torch

from conftest import launched, rel_err
from oracle import moe_oracle as O

pytestmark = pytest.mark.gpu
TOL = 2.5e-3


def _uniform(M, E, dev):
    gs = np.full(E, M // E, np.int32)
    gs[: M - int(gs.sum())] += 1
    return gs, torch.from_numpy(gs).to(dev)


def _bf16(dev, *shape, std=1.0):
    return (torch.randn(*shape, device=dev) * std).bfloat16()


f64 = lambda t: t.double().cpu().numpy()


# widths that are odd multiples of 128: 128x128 tiles, or the ring kernel's partial 256-row tiles
@pytest.mark.parametrize("M,E,N,ring", [
    (600, 2, 128, False), (4096, 8, 384, False), (4096, 8, 1408, False), (2100, 2, 6272, False),
    (16384, 8, 2176, True), (16384, 8, 640, False), (2048, 8, 12160, True), (2040, 8, 12160, False),
])
@pytest.mark.parametrize("op", ["fwd", "dlhs"])
def test_odd_multiples_of_128(dev, op, M, E, N, ring):
    from mintext_amd.kernels.grouped_matmul import _gmm_dlhs, _gmm_fwd

    K = 128
    gs, g = _uniform(M, E, dev)
    x = _bf16(dev, M, K)
    w = _bf16(dev, E, *((K, N) if op == "fwd" else (N, K)), std=0.05)
    f = _gmm_fwd if op == "fwd" else _gmm_dlhs
    names = launched(lambda: f(x, w, g))
    assert ("gmm_v3_kernel" in names, "gmm_mfma_kernel" in names) == (ring, not ring), names
    ref = O.gmm(f64(x), f64(w) if op == "fwd" else f64(w).transpose(0, 2, 1), gs)
    assert rel_err(f64(f(x, w, g)), ref) < TOL


@pytest.mark.parametrize("E,K,N,ring", [
    (8, 384, 1024, False), (32, 384, 1024, True), (32, 128, 1024, False), (3, 640, 384, False), (16, 1408, 1024, True),
])
def test_odd_multiples_of_128_tgmm(dev, E, K, N, ring):
    from mintext_amd.kernels import tgmm

    M = 40 * E + 3
    gs, g = _uniform(M, E, dev)
    gs[1], gs[0] = 0, gs[0] + gs[1]
    g = torch.from_numpy(gs).to(dev)
    x, dy = _bf16(dev, M, K), _bf16(dev, M, N)
    names = launched(lambda: tgmm(x, dy, g))
    assert ("gmm_v3_kernel" in names, "gmm_mfma_kernel" in names) == (ring, not ring), names
    assert rel_err(f64(tgmm(x, dy, g)), O.tgmm(f64(x), f64(dy), gs)) < TOL


# bf16 rows without the alignment that the bf16 tiles need: the f32 matrix tiles, single values; sums that end
# around the eights and stages of 32 that they are taken in
@pytest.mark.parametrize("K,N", [(63, 129), (33, 7), (1, 66)])
@pytest.mark.parametrize("gs", [[1, 7, 8, 9, 0, 31, 32, 33], [100, 0, 3, 65]])
def test_bf16_odd_widths(dev, K, N, gs):
    from mintext_amd.kernels import grouped_matmul, tgmm
    from mintext_amd.kernels.grouped_matmul import _gmm_dlhs

    gs = np.array(gs, np.int32)
    n, E = int(gs.sum()), len(gs)
    x, dy, w = _bf16(dev, n + 5, K), _bf16(dev, n + 5, N), _bf16(dev, E, K, N, std=0.05)
    x[n:] = dy[n:] = float("nan")
    g = torch.from_numpy(gs).to(dev)
    assert "f32mm" in launched(lambda: tgmm(x, dy, g))
    xr, dr = np.nan_to_num(f64(x)), np.nan_to_num(f64(dy))
    out, dx, dw = f64(grouped_matmul(x, w, g)), f64(_gmm_dlhs(dy, w, g)), f64(tgmm(x, dy, g))
    assert rel_err(out[:n], O.gmm(xr, f64(w), gs)[:n]) < TOL and (out[n:] == 0).all()
    assert rel_err(dx[:n], O.gmm(dr, f64(w).transpose(0, 2, 1), gs)[:n]) < TOL and (dx[n:] == 0).all()
    assert rel_err(dw, O.tgmm(xr, dr, gs)) < TOL and (dw[gs == 0] == 0).all()
