"""GPU parity of the blockwise-fp8 grouped GEMM for groups of few rows (weights streamed through
registers) at its row blocks of 16, m-tiles of 16 and 32 rows and the shortest reductions, in both
scale modes.

Against the float64 product of the dequantised operands.  bf16 outputs are rounded once (2^-9 of a
value); the f32 sums, the matrix unit's own 128-term sums and the SwiGLU's hardware exp add less than
2^-12 of the result: 2.5e-3 bounds both in the 2-norm.  A re-quantised output is within half a step of
e4m3 (2^-4 of a value at the bottom of a binade) of the bf16 one, its scale within that one's rounding
(2^-8) of amax / 448 or, in the power-of-two mode, one of the two powers next to it.
"""
from __future__ import annotations

import numpy as np
import pytest
import torch

from conftest import rel_err
from oracle import moe_oracle as O

pytestmark = pytest.mark.gpu
TOL = 2.5e-3
GROUPS = {
    "few": [1, 0, 2, 0, 0, 1, 0, 0, 3, 0, 0, 0, 1, 0, 0, 1],
    "blocks": [15, 16, 17, 0, 1, 31, 32, 33, 0, 0, 2, 0, 5, 1, 0, 0, 0, 70],
    "many": [0, 1, 2] * 200,  # more groups than a workgroup's threads
}


@pytest.mark.parametrize("scales", ["amax", "pow2"])
@pytest.mark.parametrize("groups", sorted(GROUPS))
@pytest.mark.parametrize("K,N", [(256, 256), (384, 768), (1152, 512)])
@pytest.mark.parametrize("spare", [0, 40])
def test_fp8_thin_matches_dequantised(dev, scales, groups, K, N, spare):
    from mintext_amd.kernels.fp8 import (grouped_matmul_fp8, grouped_matmul_fp8_swiglu,
                                         grouped_matmul_fp8_swiglu_gathered, quantize_fp8_rows, quantize_fp8_weights)

    gs = np.array(GROUPS[groups], np.int32)
    n, E = int(gs.sum()), len(gs)
    gen = torch.Generator(device=dev)
    gen.manual_seed(K + N)
    x = torch.randn(n + spare, K, device=dev, generator=gen) * torch.rand(n + spare, 1, device=dev, generator=gen)
    w = torch.randn(E, K, N, device=dev, generator=gen) * 0.05
    xq, xs = quantize_fp8_rows(x.bfloat16(), scales=scales)
    wq, ws = quantize_fp8_weights(w.bfloat16(), scales=scales)
    g = torch.from_numpy(gs).to(dev)
    c = lambda t: t.view(torch.uint8).cpu().numpy() if t.dtype == torch.float8_e4m3fn else t.cpu().numpy()
    h = O.gmm_fp8(c(xq), c(xs), c(wq), c(ws), gs)
    out = grouped_matmul_fp8(xq, xs, wq, ws, g, scales=scales).double().cpu().numpy()
    assert rel_err(out[:n], h[:n]) < TOL and (out[n:] == 0).all()

    yq, ys, yb = grouped_matmul_fp8_swiglu(xq, xs, wq, ws, g, return_bf16=True, scales=scales)
    i = N // 2
    want = h[:, :i] / (1 + np.exp(-h[:, :i])) * h[:, i:]
    b = yb.double().cpu().numpy()
    assert rel_err(b[:n], want[:n]) < TOL and (b[n:] == 0).all()
    s = ys.double().cpu().numpy()
    deq = yq.double().cpu().numpy().reshape(n + spare, i // 128, 128) * s[..., None]
    blk = b.reshape(n + spare, i // 128, 128)
    amax = np.abs(blk).max(-1)
    assert (np.abs(deq - blk) <= np.abs(blk) * (2.0 ** -4 + 2.0 ** -8) + s[..., None] * 2.0 ** -9).all()
    ratio = np.where(amax > 0, s / np.where(amax > 0, amax / 448.0, 1), 1)
    if scales == "amax":
        assert (np.abs(ratio - 1) <= 2.0 ** -8).all()
    else:
        assert (ratio >= 1 - 2.0 ** -8).all() and (ratio <= 2 * (1 + 2.0 ** -8)).all()
    assert (s[n:] == 1).all()
    # the gathered form: the same rows in another order, same bits
    perm = torch.randperm(n + spare, device=dev, generator=gen)
    si = torch.argsort(perm).to(torch.int32)
    gq, gsc = grouped_matmul_fp8_swiglu_gathered(xq.view(torch.uint8)[perm].view(torch.float8_e4m3fn), xs[perm], si, 1,
                                                 wq, ws, g, scales=scales)
    assert torch.equal(gq.view(torch.uint8), yq.view(torch.uint8)) and torch.equal(gsc, ys)
