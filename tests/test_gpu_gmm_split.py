"""GPU parity of the grouped GEMM's split tail around the shortest reduction that splits, at the one, two
and four pieces that the dispatch can choose, alone and behind rounds of whole tiles (where pieces are
taken by ticket, on any XCD), with reductions that end inside a stage, and with last tiles of every
height, against the same tiles computed whole.

The two differ only in how a tile's f32 sum is associated, so by at most one step of bf16: its
spacing is 2^-7 of a value at the bottom of a binade (8 significant bits) and less elsewhere.  Values
that cancel to less than the f32 sums' own error may differ by that, 2^-16 of the largest value.
"""
from __future__ import annotations

import pytest
import torch

from conftest import split_pieces, tile_list_workspace_bytes

pytestmark = pytest.mark.gpu


def _check(dev, op, gs, Kred, N, few_stages):
    from mintext_amd import _lib as L

    gen = torch.Generator(device=dev)
    gen.manual_seed(Kred + N)
    M, E = sum(gs), len(gs)
    pieces = split_pieces(sum(-(-n // 256) for n in gs), -(-N // 256), Kred // 32, few_stages)
    gs = torch.tensor(gs, dtype=torch.int32, device=dev)
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
    # some of the f32 sums round to another bf16 value when they are added in pieces
    assert torch.equal(split, whole) == (pieces == 1)
    for _ in range(3):
        assert torch.equal(call(full), split)  # summed in piece order, whatever the order of arrival
    assert ((split - whole).abs() <= whole.abs() * 2.0 ** -7 + whole.abs().max() * 2.0 ** -16).all()
    return pieces


@pytest.mark.parametrize("op", ["fwd", "dlhs"])
@pytest.mark.parametrize("M,E,Kred,N,pieces", [
    (300, 2, 1248, 1024, 1),    # 39 stages: too short for two pieces
    (300, 2, 1280, 1024, 2),    # few tiles: 40 stages in two pieces
    (300, 2, 2560, 1024, 4),    # the wave rows of some pieces empty
    (1100, 2, 2592, 2048, 4),   # pieces of unequal length
    (700, 3, 5120, 512, 4),
    (300, 2, 2568, 1032, 4),    # widths that are multiples of 8: the last piece ends inside a stage
    (700, 3, 5128, 520, 4),
    (8000, 32, 2560, 2560, 2),  # behind a round of whole tiles
    (8000, 32, 2568, 2568, 2),
])
def test_split_tail_equals_whole_tiles(dev, op, M, E, Kred, N, pieces):
    gs = [M // E - 7] + [M // E] * (E - 1)
    assert _check(dev, op, gs, Kred, N, 16) == pieces


# groups of over 512 rows: the one-wave-per-SIMD kernel; last tiles of 32, 64, 96, 128 and 256 rows, which
# differ in how a piece is read back
@pytest.mark.parametrize("op", ["fwd", "dlhs"])
@pytest.mark.parametrize("gs,Kred,N,pieces", [
    ([512 + 30, 512 + 61], 2112, 1024, 2),
    ([512 + 90, 512 + 121], 5184, 1024, 4),
    ([1043, 1050], 5184, 1024, 4),
    # 33 to 48 tiles an XCD: whole rounds, then pieces taken by ticket (16 n-tiles: those split over the XCDs)
    ([2400, 2330], 2560, 4096, 2),
    ([2400, 2330], 5120, 4352, 2),
    ([2080] * 4, 5120, 2304, 3),
    ([1550, 1570, 1600, 1630], 5120, 2560, 4),
])
def test_split_tail_one_wave_per_simd(dev, op, gs, Kred, N, pieces):
    assert _check(dev, op, gs, Kred, N, 32) == pieces
