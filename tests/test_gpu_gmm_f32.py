"""GPU parity of the f32 grouped GEMMs (f32 matrix cores, 64x64 tiles, 32-deep stages) at the edges of
their tiles and stages, aligned and not, and of bf16 at widths that are no multiple of 8, which run on
the same tiles.

Against the float64 oracle.  f32: the sums' rounding is at most about 2^-24 * sqrt(K) of the sum of the
products' magnitudes, itself about sqrt(K) of the result for random signs: K * 2^-24 <= 8e-6 in the
2-norm at K <= 129.  bf16: one rounding of the output, 2^-9, more.
"""
from __future__ import annotations

import numpy as np
import pytest
import torch

from conftest import rel_err
from oracle import moe_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,tol", [("f32", 8e-6), ("bf16", 2.5e-3)])
@pytest.mark.parametrize("groups", [[1, 0, 64, 65, 3], [0, 200, 31, 32, 33]])
@pytest.mark.parametrize("Kin,Kout", [(1, 2), (33, 62), (36, 68), (64, 130), (129, 64)])
def test_f32_tiles_match_oracle(dev, dtype, tol, groups, Kin, Kout):
    from mintext_amd.kernels import grouped_matmul, tgmm
    from mintext_amd.kernels.grouped_matmul import _gmm_dlhs, grouped_matmul_swiglu

    dt = torch.float32 if dtype == "f32" else torch.bfloat16
    gs, spare = np.array(groups, np.int32), 3
    n = int(gs.sum())
    gen = torch.Generator(device=dev)
    gen.manual_seed(Kin + Kout)
    r = lambda *shape: torch.randn(*shape, device=dev, generator=gen).to(dt)
    x, w, grad = r(n + spare, Kin), r(len(gs), Kin, Kout), r(n + spare, Kout)
    x[n:] = grad[n:] = float("nan")  # rows of no group reach no output
    g = torch.from_numpy(gs).to(dev)
    f = lambda t: np.nan_to_num(t.double().cpu().numpy())
    h = O.gmm(f(x), f(w), gs)
    out = grouped_matmul(x, w, g).double().cpu().numpy()
    assert rel_err(out[:n], h[:n]) < tol and (out[n:] == 0).all()
    dx = _gmm_dlhs(grad, w, g).double().cpu().numpy()
    assert rel_err(dx[:n], O.gmm(f(grad), f(w).transpose(0, 2, 1), gs)[:n]) < tol and (dx[n:] == 0).all()
    dw = tgmm(x, grad, g).double().cpu().numpy()
    assert rel_err(dw, O.tgmm(f(x), f(grad), gs)) < tol and (dw[gs == 0] == 0).all()
    y = grouped_matmul_swiglu(x, w, g).double().cpu().numpy()
    i = Kout // 2
    assert rel_err(y[:n], (h[:, :i] / (1 + np.exp(-h[:, :i])) * h[:, i:])[:n]) < tol and (y[n:] == 0).all()
