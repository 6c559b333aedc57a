"""GPU parity of the bf16 grouped GEMMs at widths that are multiples of 8 but of no tile: n-tiles and
dW tiles that hang over the last column or row, reductions that end inside a ring stage.

Against the float64 oracle on the same bf16 operands.  The output is rounded once (relative error at
most 2^-9 per value, so at most 2^-9 in the 2-norm); the f32 accumulation adds about 2^-24 * sqrt(K) of
the sum of the products' magnitudes, below 2^-15 of the result here: 2.5e-3 bounds both.  Rows past
sum(group_sizes) hold NaN: they may reach no output.
"""
from __future__ import annotations

import numpy as np
import pytest
import torch

from conftest import rel_err
from oracle import moe_oracle as O

pytestmark = pytest.mark.gpu
TOL = 2.5e-3

# (Kin, Kout): one chunk; a chunk past a stage / a tile; a chunk short of one; a 32- but not 64-multiple
WIDTHS = [(8, 8), (40, 264), (24, 248), (96, 136), (264, 520), (1000, 704), (704, 1536)]


def _case(M, E, Kin, Kout, dev, spare=5):
    rng = np.random.default_rng(Kin * 1000 + Kout)
    gs = rng.multinomial(M - spare, rng.dirichlet(np.full(E, 0.5)))
    gs[E // 2] = 0
    x = torch.randn(M, Kin, device=dev).bfloat16()
    x[int(gs.sum()):] = float("nan")
    w = (torch.randn(E, Kin, Kout, device=dev) * 0.05).bfloat16()
    return gs.astype(np.int32), x, w


def _f64(t):
    return t.double().cpu().numpy()


@pytest.mark.parametrize("M,E", [(37, 3), (900, 4)])
@pytest.mark.parametrize("Kin,Kout", WIDTHS)
def test_edge_widths_match_oracle(dev, M, E, Kin, Kout):
    from mintext_amd.kernels import grouped_matmul, tgmm
    from mintext_amd.kernels.grouped_matmul import _gmm_dlhs, grouped_matmul_swiglu

    gs, x, w = _case(M, E, Kin, Kout, dev)
    n = int(gs.sum())
    g = torch.from_numpy(gs).to(dev)
    xr = np.nan_to_num(_f64(x))
    h = O.gmm(xr, _f64(w), gs)
    out = _f64(grouped_matmul(x, w, g))
    assert rel_err(out[:n], h[:n]) < TOL and (out[n:] == 0).all()
    grad = torch.randn(M, Kout, device=dev).bfloat16()
    grad[n:] = float("nan")
    gr = np.nan_to_num(_f64(grad))
    dx = _f64(_gmm_dlhs(grad, w, g))
    assert rel_err(dx[:n], O.gmm(gr, _f64(w).transpose(0, 2, 1), gs)[:n]) < TOL and (dx[n:] == 0).all()
    dw = _f64(tgmm(x, grad, g))
    assert rel_err(dw, O.tgmm(xr, gr, gs)) < TOL and (dw[gs == 0] == 0).all()
    if Kout % 16 == 0:
        y = _f64(grouped_matmul_swiglu(x, w, g))
        i = Kout // 2
        want = h[:, :i] / (1 + np.exp(-h[:, :i])) * h[:, i:]
        assert rel_err(y[:n], want[:n]) < TOL and (y[n:] == 0).all()
