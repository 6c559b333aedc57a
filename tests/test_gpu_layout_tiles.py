"""Whole-tile transposes (mtx_transpose_batched) and weight quantisation at the edges of their variants:
tile remainders (which take the general kernel), wave counts that do not fill a workgroup, fused halves
with their own strides, and both sides of the size at which the data is streamed past the caches.
Transposes are exact; the quantiser's two variants give the same bytes."""
from __future__ import annotations

import pytest
import torch


def _transpose(x, out, R, C, out_bs, out_ld, offset=0):
    from mintext_amd import _lib

    rc = _lib.lib().mtx_transpose_batched(
        x.data_ptr(), _lib.dtype_code(x.dtype), x.shape[0], R, C, x.stride(0), x.stride(1),
        out.data_ptr() + offset * out.element_size(), out_bs, out_ld, _lib.stream(x.device))
    assert rc == 0


@pytest.mark.gpu
@pytest.mark.parametrize("B,R,C", [
    (1, 32, 32), (1, 64, 64), (3, 64, 192), (2, 320, 64), (2, 192, 320), (2, 96, 160), (2, 72, 64), (2, 64, 72),
    (16, 1024, 2048), (33, 1024, 1024),  # 67 and 69 MB in and out for bf16, 134 and 138 MB for f32
    (64, 1024, 1024),  # 268 MB in and out for bf16: streamed
    (5500, 64, 192), (2800, 96, 160),  # streamed, 3 (bf16) and 15 (f32) wave tiles: the last workgroup partly empty
])
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
def test_transpose_tiles(dev, B, R, C, dt):
    torch.manual_seed(B + R + C)
    x = torch.randn(B, R, C + 8, device=dev).to(dt)[:, :, :C]  # rows longer than the tile's columns
    out = torch.full((B, C, 2 * R), 7.0, device=dev, dtype=dt)
    _transpose(x, out, R, C, C * 2 * R, 2 * R, offset=R)  # the second half of a fused tensor
    assert torch.equal(out[:, :, R:], x.transpose(1, 2))
    assert bool((out[:, :, :R] == 7.0).all())


@pytest.mark.gpu
@pytest.mark.parametrize("pow2", [False, True])
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
def test_streamed_weight_codes(dev, dt, pow2):
    from mintext_amd import _lib

    torch.manual_seed(5)
    E, K, N = 48, 1024, 1024  # 151 MB (bf16) of weights and codes in one call; an expert alone is 3 MB
    w = torch.randn(E, K, N, device=dev).to(dt)
    f = _lib.lib().mtx_quant_fp8_weights_p2 if pow2 else _lib.lib().mtx_quant_fp8_weights

    def quant(w):
        q = torch.zeros(w.shape[0], N, K, device=dev, dtype=torch.uint8)
        s = torch.zeros(w.shape[0], N // 128, K // 128, device=dev)
        rc = f(w.data_ptr(), _lib.dtype_code(dt), w.shape[0], K, N, q.data_ptr(), s.data_ptr(),
               _lib.stream(w.device))
        assert rc == 0
        return q, s

    q, s = quant(w)
    for e in (0, 17, 47):
        qe, se = quant(w[e:e + 1])
        assert torch.equal(q[e], qe[0]) and torch.equal(s[e], se[0])
