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


# ---- groups of few rows: which kernel, by the group sizes ----------------------------------------------------

def _concentrated(M, E, k):
    gs = np.zeros(E, np.int32)
    gs[E // 2:E // 2 + k] = M // k
    gs[E // 2] += M - M // k * k
    return gs


# "few": the few-row kernel alone; "spread" / "concentrated": both are launched and the group sizes decide
# (the kernel that has the call is the one whose tiles are computed: the tile list is empty otherwise)
FEW = [
    # M (three rows of no group), E, K, N (SwiGLU: gate and up columns), SwiGLU, launches with rows spread, launches on few groups
    (16, 8, 4096, 1024, False, "few", "few"),
    (256, 64, 512, 2048, False, "few", "few"),
    (512, 64, 512, 2048, False, "both", "both"),
    (512, 64, 512, 1000, False, "few", "few"),
    (512, 64, 512, 1032, False, "both", "both"),      # a ring kernel with partial tiles beside it
    (128, 32, 256, 2048, True, "few", "few"),
    (256, 32, 256, 2048, True, "ring", "ring"),        # SwiGLU: less than 128 MB of weights
    (256, 32, 1024, 2048, True, "both", "both"),
    (130, 32, 1032, 2064, True, "both", "both"),
    (512, 128, 64, 5120, False, "ring", "ring"),       # a grid of more than 4096 workgroups
    (12, 4, 8448, 512, False, "ring", "ring"),         # a long plain reduction: too few tiles for the chip
    (64, 64, 4160, 512, False, "both", "both"),
]


@pytest.mark.parametrize("M,E,K,N,swiglu,spread,concentrated", FEW)
def test_few_rows_by_group_sizes(dev, M, E, K, N, swiglu, spread, concentrated):
    from mintext_amd.kernels.grouped_matmul import _gmm_fwd, grouped_matmul_swiglu

    f = grouped_matmul_swiglu if swiglu else _gmm_fwd
    w = _bf16(dev, E, K, N, std=0.05)
    w64 = f64(w)
    for gs, want in ((_uniform(M - 3, E, dev)[0], spread), (_concentrated(M - 3, E, 1), concentrated),
                     (_concentrated(M - 3, E, 2), concentrated), (np.zeros(E, np.int32), concentrated)):
        x = _bf16(dev, M, K)
        n = int(gs.sum())
        g = torch.from_numpy(gs).to(dev)
        names = launched(lambda: f(x, w, g))
        assert ("gmm_thin" in names, "gmm_v3" in names) == (want != "ring", want != "few"), names
        h = O.gmm(f64(x), w64, gs)
        i = N // 2
        ref = h[:, :i] / (1 + np.exp(-h[:, :i])) * h[:, i:] if swiglu else h
        out = f64(f(x, w, g))
        assert rel_err(out[:n], ref[:n]) < TOL and (out[n:] == 0).all()


@pytest.mark.parametrize("scales", ["amax", "pow2"])
@pytest.mark.parametrize("M,E,K,N,want", [(256, 64, 256, 2048, "few"), (512, 64, 256, 2048, "both"), (24, 2, 256, 32768, "both")])
def test_fp8_few_rows_by_group_sizes(dev, scales, M, E, K, N, want):
    from mintext_amd.kernels.fp8 import (grouped_matmul_fp8, grouped_matmul_fp8_swiglu, quantize_fp8_rows,
                                         quantize_fp8_weights)

    xq, xs = quantize_fp8_rows(_bf16(dev, M, K), scales=scales)
    wq, ws = quantize_fp8_weights(_bf16(dev, E, K, N, std=0.05), scales=scales)
    c = lambda t: t.view(torch.uint8).cpu().numpy() if t.dtype == torch.float8_e4m3fn else t.cpu().numpy()
    for gs in (_uniform(M - 3, E, dev)[0], _concentrated(M - 3, E, 1), _concentrated(M - 3, E, 2), np.zeros(E, np.int32)):
        n = int(gs.sum())
        g = torch.from_numpy(gs).to(dev)
        f = lambda: grouped_matmul_fp8(xq, xs, wq, ws, g, scales=scales)
        names = launched(f)
        assert ("gmm_fp8_thin" in names, "gmm_fp8_v4" in names) == (True, want == "both"), names
        h = O.gmm_fp8(c(xq), c(xs), c(wq), c(ws), gs)
        out = f64(f())
        assert rel_err(out[:n], h[:n]) < TOL and (out[n:] == 0).all()
        _, ys, yb = grouped_matmul_fp8_swiglu(xq, xs, wq, ws, g, return_bf16=True, scales=scales)
        i = N // 2
        b = f64(yb)
        assert rel_err(b[:n], (h[:, :i] / (1 + np.exp(-h[:, :i])) * h[:, i:])[:n]) < TOL and (b[n:] == 0).all()
        assert (f64(ys)[n:] == 1).all()


@pytest.mark.parametrize("fp8", [False, True])
def test_few_rows_choice_under_capture(dev, fp8):
    """A captured call chooses again in each replay, from the group sizes it finds."""
    from mintext_amd.kernels.fp8 import grouped_matmul_fp8, quantize_fp8_rows, quantize_fp8_weights
    from mintext_amd.kernels.grouped_matmul import grouped_matmul
    from mintext_amd.moe import CapturedLayer

    M, E, K, N = 512, 64, 256, 2048
    x, w = _bf16(dev, M, K), _bf16(dev, E, K, N, std=0.05)
    if fp8:
        (xq, xs), (wq, ws) = quantize_fp8_rows(x), quantize_fp8_weights(w)
        f = lambda g: grouped_matmul_fp8(xq, xs, wq, ws, g)
    else:
        f = lambda g: grouped_matmul(x, w, g)
    spread, few = _uniform(M - 3, E, dev)[1], torch.from_numpy(_concentrated(M - 3, E, 1)).to(dev)
    layer = CapturedLayer(f, spread.clone())
    for g in (spread, few, few, spread, torch.zeros_like(few), few):
        layer.inputs[0].copy_(g)
        got = layer.replay().clone()
        torch.cuda.synchronize()
        assert torch.equal(got, f(g))


# ---- the few-row kernel's wide SwiGLU form (from 512 MB of weights over its m-tiles): 128 gate columns in one half
# of the waves, the matching up columns in the other; partial columns, a reduction that ends inside a chunk
@pytest.mark.parametrize("M", [15, 60])
def test_few_rows_wide_form(dev, M):
    _wide(dev, M, 16, 1032, 7304, 4)


@pytest.mark.parametrize("M,K,I", [(13, 8968, 1032), (32, 4840, 1544)])
def test_few_rows_wide_form_eight_waves(dev, M, K, I):
    _wide(dev, M, 16, K, I, 8)


def _wide(dev, M, E, K, I, waves):
    from mintext_amd.kernels.grouped_matmul import grouped_matmul_swiglu

    gs, g = _uniform(M, E, dev)
    x = _bf16(dev, M + 1, K)
    x[M] = float("nan")
    w = torch.empty(E, K, 2 * I, dtype=torch.bfloat16, device=dev).normal_(0.0, 0.02)
    names = launched(lambda: grouped_matmul_swiglu(x, w, g))
    tb = 1 if M + 1 <= 2 * E else 2
    assert f"gmm_thin_kernel<2, {tb}, {waves}," in names, names
    y = grouped_matmul_swiglu(x, w, g)
    ref = torch.zeros(M, I, dtype=torch.float64, device=dev)
    r = 0
    for e in range(E):
        h = x[r:r + int(gs[e])].double() @ w[e].double()
        ref[r:r + int(gs[e])] = torch.nn.functional.silu(h[:, :I]) * h[:, I:]
        r += int(gs[e])
    assert rel_err(f64(y[:M]), ref.cpu().numpy()) < TOL and (y[M] == 0).all()


# ---- outputs off a 16-byte boundary, which only a caller of the C interface has: 128x128 tiles at any size where
# the width is a multiple of 128, else single values
@pytest.mark.parametrize("op", ["fwd", "dlhs", "tgmm"])
@pytest.mark.parametrize("N", [640, 264])
def test_outputs_at_any_offset(dev, op, N):
    from mintext_amd import _lib as L

    E, K, M = 4, 128, 4 * 512
    if op == "tgmm":
        E, K, N = 16, N if N % 128 else 1408, 1024
        M = 40 * E
    gs, g = _uniform(M, E, dev)
    x, y = _bf16(dev, M, K), _bf16(dev, M, N)
    w = _bf16(dev, E, *((K, N) if op == "fwd" else (N, K)), std=0.05)
    n = E * K * N if op == "tgmm" else M * N
    ws = L.workspace(L.query("mtx_gmm_workspace_size", M, E), dev)
    tail = (ws.data_ptr(), ws.numel(), L.stream(dev))
    outs = []
    for offset in (0, 1):
        buf = torch.full((n + offset,), float("nan"), device=dev, dtype=torch.bfloat16)
        out = buf[offset:]
        if op == "tgmm":
            f = lambda: L.call("mtx_tgmm", L.ptr(x), L.ptr(y), L.ptr(g), L.MTX_BF16, M, K, N, E, out.data_ptr(), *tail)
        else:
            kin, kout = (K, N) if op == "fwd" else (N, K)
            code = L.MTX_GMM_OP_FWD if op == "fwd" else L.MTX_GMM_OP_DLHS
            f = lambda: L.call("mtx_gmm_tiled", code, L.ptr(x), L.ptr(w), L.ptr(g), L.MTX_BF16, M, kin, kout, E, 0, 0,
                               out.data_ptr(), *tail)
        names = launched(f)
        if offset:
            assert ("gmm_mfma" if N % 128 == 0 and K % 128 == 0 else "f32mm") in names, names
        outs.append(f64(out))
    if op == "tgmm":
        ref = O.tgmm(f64(x), f64(y), gs).ravel()
    else:
        ref = O.gmm(f64(x), f64(w) if op == "fwd" else f64(w).transpose(0, 2, 1), gs).ravel()
    for o in outs:
        assert rel_err(o, ref) < TOL
