"""GPU parity of the bf16 grouped GEMM for groups of few rows (weights streamed through registers), at
its row blocks of 16, m-tiles of 16 and 32 rows, chunks of 32 k, and 64- and 128-column tiles.

Against the float64 oracle on the same bf16 operands, with the bound of one bf16 rounding (2^-9 of a
value) plus the f32 sums (below 2^-15 of the result at these lengths): 2.5e-3 in the 2-norm.  Rows
past sum(group_sizes) hold NaN and may reach no output.
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
    "few": [1, 0, 2, 0, 0, 1, 0, 0, 3, 0, 0, 0, 1, 0, 0, 1],                  # 16-row m-tiles
    "blocks": [15, 16, 17, 0, 1, 31, 32, 33, 0, 0, 2, 0, 5, 1, 0, 0, 0, 70],  # 32-row m-tiles, several in a group
    "many": [0, 1, 2] * 100,                                                  # more groups than a workgroup's threads
}


@pytest.mark.parametrize("groups", sorted(GROUPS))
@pytest.mark.parametrize("Kin,Kout", [(8, 16), (40, 136), (64, 256), (264, 400), (1056, 768)])
@pytest.mark.parametrize("spare", [0, 40])
def test_thin_matches_oracle(dev, groups, Kin, Kout, spare):
    from mintext_amd.kernels import grouped_matmul
    from mintext_amd.kernels.grouped_matmul import grouped_matmul_swiglu

    gs = np.array(GROUPS[groups], np.int32)
    n = int(gs.sum())
    gen = torch.Generator(device=dev)
    gen.manual_seed(Kin + Kout)
    x = torch.randn(n + spare, Kin, device=dev, generator=gen).bfloat16()
    x[n:] = float("nan")
    w = (torch.randn(len(gs), Kin, Kout, device=dev, generator=gen) * 0.05).bfloat16()
    g = torch.from_numpy(gs).to(dev)
    h = O.gmm(np.nan_to_num(x.double().cpu().numpy()), w.double().cpu().numpy(), gs)
    out = grouped_matmul(x, w, g).double().cpu().numpy()
    assert rel_err(out[:n], h[:n]) < TOL and (out[n:] == 0).all()
    y = grouped_matmul_swiglu(x, w, g).double().cpu().numpy()
    i = Kout // 2
    assert rel_err(y[:n], (h[:, :i] / (1 + np.exp(-h[:, :i])) * h[:, i:])[:n]) < TOL and (y[n:] == 0).all()


@pytest.mark.parametrize("T,E,K", [(1, 64, 8), (37, 8, 2), (90, 32, 4)])
def test_thin_gathered_equals_sorted(dev, T, E, K):
    from mintext_amd.kernels import route, route_topk
    from mintext_amd.kernels.grouped_matmul import grouped_matmul_swiglu, grouped_matmul_swiglu_gathered

    gen = torch.Generator(device=dev)
    gen.manual_seed(T)
    x = torch.randn(T, 192, device=dev, generator=gen).bfloat16()
    w = (torch.randn(E, 192, 512, device=dev, generator=gen) * 0.05).bfloat16()
    idx, _ = route_topk(torch.randn(T, E, device=dev, generator=gen), K)
    st, si, gs = route(x, idx, E)
    assert torch.equal(grouped_matmul_swiglu_gathered(x, si, K, w, gs), grouped_matmul_swiglu(st, w, gs))
