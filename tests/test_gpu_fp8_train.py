"""The fused fp8 training step equals its separate steps (route, fp8 GEMMs, SwiGLU, combine and their
VJPs) bit for bit, outputs and gradients: the same codes, scales and products, made by fewer kernels.
Groups around the 128-row chunks, empty groups, ids of no expert, both scale modes, partial gradients."""
from __future__ import annotations

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _steps(x, idx, w, gate_up, down, scales):
    from mintext_amd.kernels.fp8 import grouped_matmul_fp8_vjp
    from mintext_amd.kernels.moe_dispatch import route, unroute
    from mintext_amd.kernels.swiglu import swiglu_autograd

    st, si, gs = route(x, idx, gate_up.shape[0])
    h = grouped_matmul_fp8_vjp(st, gate_up, gs, scales=scales)
    out = grouped_matmul_fp8_vjp(swiglu_autograd(h), down, gs, scales=scales)
    return unroute(out, si, w, idx.shape[1])


def _inputs(dev, T, D, E, K, I, wdt, invalid=False):
    rng = np.random.default_rng(T + E)
    # a popular expert, experts with a row or none, the rest around a chunk
    p = rng.dirichlet(np.full(E, 0.3))
    idx = np.stack([rng.choice(E, K, replace=False, p=(p + 1e-6) / (p + 1e-6).sum()) for _ in range(T)]).astype(np.int32)
    if invalid:
        idx[rng.random(idx.shape) < 0.05] = -1
    gen = torch.Generator(device=dev)
    gen.manual_seed(T)
    r = lambda *s: torch.randn(*s, device=dev, generator=gen)
    return (r(T, D).bfloat16(), torch.from_numpy(idx).to(dev), torch.rand(T, K, device=dev, generator=gen),
            (r(E, D, 2 * I) * 0.05).to(wdt), (r(E, I, D) * 0.05).to(wdt), r(T, D))


@pytest.mark.parametrize("scales", ["amax", "pow2"])
@pytest.mark.parametrize("T,D,E,K,I,wdt,invalid", [
    (1, 256, 4, 2, 256, torch.bfloat16, False),
    (128, 512, 3, 1, 256, torch.bfloat16, False),
    (333, 256, 9, 3, 512, torch.float32, False),
    (1500, 768, 12, 4, 256, torch.bfloat16, True),
])
def test_fused_step_equals_separate_steps(dev, scales, T, D, E, K, I, wdt, invalid):
    from mintext_amd.kernels.fp8_train import experts_fp8_train, experts_fp8_train_supported

    *t, dout = _inputs(dev, T, D, E, K, I, wdt, invalid)
    assert experts_fp8_train_supported(*t, scales)
    got = []
    for f in (_steps, experts_fp8_train):
        x, idx, w, gu, dn = (a.clone() for a in t)
        leaves = [a.requires_grad_(True) for a in (x, w, gu, dn)]
        out = f(x, idx, w, gu, dn, scales)
        got.append((out, *torch.autograd.grad(out, leaves, dout)))
    for a, b in zip(*got):
        assert a.dtype == b.dtype and torch.equal(a, b)


@pytest.mark.parametrize("needs", [(1, 0, 0, 0), (0, 1, 0, 0), (0, 0, 1, 0), (0, 0, 0, 1), (1, 0, 0, 1), (0, 1, 1, 0)])
def test_partial_gradients(dev, needs):
    from mintext_amd.kernels.fp8_train import experts_fp8_train

    *t, dout = _inputs(dev, 200, 256, 5, 2, 256, torch.bfloat16)
    got = []
    for f in (_steps, experts_fp8_train):
        x, idx, w, gu, dn = (a.clone() for a in t)
        leaves = [a.requires_grad_(True) for a, n in zip((x, w, gu, dn), needs) if n]
        out = f(x, idx, w, gu, dn, "pow2")
        got.append((out, *torch.autograd.grad(out, leaves, dout)))
    for a, b in zip(*got):
        assert torch.equal(a, b)


def test_no_gradient_and_changed_weights(dev):
    from mintext_amd.moe import moe_experts_forward_fp8_train

    x, idx, w, gu, dn, dout = _inputs(dev, 64, 256, 4, 2, 256, torch.bfloat16)
    with torch.no_grad():
        plain = moe_experts_forward_fp8_train(x, idx, w, gu, dn)
    assert not plain.requires_grad and torch.equal(plain, _steps(x, idx, w, gu, dn, "amax"))
    gu.requires_grad_(True)
    out = moe_experts_forward_fp8_train(x, idx, w, gu, dn)
    with torch.no_grad():
        gu.mul_(2.0)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        out.backward(dout)


@pytest.mark.parametrize("offset", [1, 4, 8])
def test_tokens_at_any_offset(dev, offset):
    """Tokens that start off a 16-byte boundary take the separate steps, whose sorted copy is aligned."""
    from mintext_amd.kernels.fp8_train import experts_fp8_train_supported
    from mintext_amd.moe import moe_experts_forward_fp8_train

    x, idx, w, gu, dn, _ = _inputs(dev, 65, 256, 4, 2, 256, torch.bfloat16)
    moved = torch.empty(x.numel() + offset, dtype=x.dtype, device=dev)[offset:].view(x.shape)
    moved.copy_(x)
    assert experts_fp8_train_supported(moved, idx, w, gu, dn, "amax") == (offset == 8)
    got = moe_experts_forward_fp8_train(moved, idx, w, gu, dn, scales="amax")
    assert torch.equal(got, moe_experts_forward_fp8_train(x, idx, w, gu, dn, scales="amax"))


# few rows per expert (the codes' padding to 128 rows outweighs them), many, a token per row; every choice of
# what is kept
@pytest.mark.parametrize("T,D,E,K,I,wdt", [
    (96, 512, 16, 2, 256, torch.bfloat16), (4096, 512, 8, 4, 256, torch.bfloat16), (2048, 512, 8, 1, 512, torch.float32),
    (8192, 256, 2, 1, 256, torch.bfloat16), (1024, 1024, 4, 2, 1024, torch.bfloat16),
])
def test_memory_of_fused_step(dev, T, D, E, K, I, wdt):
    """Between its passes, and at the peak of both, a layer holds no more than the separate steps do."""
    from mintext_amd.kernels.fp8_train import experts_fp8_train

    *t, dout = _inputs(dev, T, D, E, K, I, wdt)
    used = {}
    for f in (_steps, experts_fp8_train, _steps, experts_fp8_train):  # the first two also warm the allocator
        x, idx, w, gu, dn = (a.clone() for a in t)
        leaves = [a.requires_grad_(True) for a in (x, w, gu, dn)]
        torch.cuda.synchronize()
        torch.cuda.reset_peak_memory_stats()
        base = torch.cuda.memory_allocated()
        out = f(x, idx, w, gu, dn, "amax")
        held = torch.cuda.memory_allocated() - base
        grads = torch.autograd.grad(out, leaves, dout)
        used[f] = (held, torch.cuda.max_memory_allocated() - base)
        del out, grads
    slack = 1 << 16  # the allocator rounds each tensor up to 512 bytes
    for a, b in zip(used[experts_fp8_train], used[_steps]):
        assert a <= b + slack, used


def test_tokens_changed_before_the_backward(dev):
    """The gradients are of the tokens that the forward saw, as in the separate steps."""
    from mintext_amd.kernels.fp8_train import experts_fp8_train

    *t, dout = _inputs(dev, 200, 256, 5, 2, 256, torch.bfloat16)
    got = []
    for change in (False, True):
        x, idx, w, gu, dn = (a.clone() for a in t)
        gu.requires_grad_(True)
        out = experts_fp8_train(x, idx, w, gu, dn, "amax")
        if change:
            x.zero_()
        got.append(torch.autograd.grad(out, gu, dout)[0])
    assert torch.equal(*got)
