"""GPU parity of the grouped GEMM's split tail around the shortest reduction that splits, and at the
one, two and four pieces that the dispatch can choose, against the same tiles computed whole.

The two differ only in how a tile's f32 sum is associated, so by at most one step of bf16: its
spacing is 2^-7 of a value at the bottom of a binade (8 significant bits) and less elsewhere.  Values
that cancel to less than the f32 sums' own error may differ by that, 2^-16 of the largest value.
"""
from __future__ import annotations

import pytest
import torch

from conftest import tile_list_workspace_bytes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("op", ["fwd", "dlhs"])
@pytest.mark.parametrize("M,E,Kred,N", [
    (300, 2, 1248, 1024),    # 39 stages: too short for two pieces
    (300, 2, 1280, 1024),    # few tiles: 40 stages in two pieces
    (300, 2, 2560, 1024),    # two pieces, the wave rows of some of them empty
    (1100, 2, 2592, 2048),   # pieces of unequal length
    (700, 3, 5120, 512),     # four pieces
    (2100, 2, 5184, 1024),   # groups of over 512 rows: the one-wave-per-SIMD kernel
])
def test_split_tail_equals_whole_tiles(dev, op, M, E, Kred, N):
    from mintext_amd import _lib as L

    gen = torch.Generator(device=dev)
    gen.manual_seed(Kred + N)
    gs = torch.tensor([M // E - 7] + [M // E] * (E - 1), dtype=torch.int32, device=dev)
    a = torch.randn(M, Kred, device=dev, generator=gen).bfloat16()
    shape = (E, Kred, N) if op == "fwd" else (E, N, Kred)
    w = (torch.randn(*shape, device=dev, generator=gen) * 0.05).bfloat16()
    kin, kout = shape[1:]
    code = L.MTX_GMM_OP_FWD if op == "fwd" else L.MTX_GMM_OP_DLHS
    full = L.query("mtx_gmm_workspace_size", M, E)

    def call(nbytes):
        out = torch.full((M, N), float("nan"), device=dev, dtype=torch.bfloat16)
        ws = torch.full((nbytes,), 0xAB, dtype=torch.uint8, device=dev)
        L.call("mtx_gmm_tiled", code, L.ptr(a), L.ptr(w), L.ptr(gs), L.MTX_BF16, M, kin, kout, E, 256, 0, L.ptr(out),
               L.ptr(ws), nbytes, L.stream(dev))
        return out.double()

    whole = call(tile_list_workspace_bytes(M, E))
    split = call(full)
    again = call(full)
    # some of the f32 sums round to another bf16 value when they are added in pieces
    assert torch.equal(split, whole) == (Kred < 1280)
    assert torch.equal(split, again)  # summed in piece order, whatever the order of arrival
    assert ((split - whole).abs() <= whole.abs() * 2.0 ** -7 + whole.abs().max() * 2.0 ** -16).all()
