"""When the ops may run without their autograd Functions: not while something is active that has to see them."""
from __future__ import annotations

import pytest
import torch

from mintext_amd import _lib as L


def _traced(f, *args):
    return torch.jit.trace(f, args, check_trace=False)


def test_plain_forward_conditions():
    x, g = torch.ones(2), torch.ones(2, requires_grad=True)
    assert L.plain_forward(x) and not L.plain_forward(x, g)
    assert L.plain_forward(x, None) and not L.plain_forward(None, g)  # an operand that is not given
    with torch.no_grad():
        assert L.plain_forward(x, g)
    with torch.autograd.forward_ad.dual_level():
        assert not L.plain_forward(x)
    seen = []

    def f(a):
        seen.append(L.plain_forward(a))
        return a * 2

    torch.func.vmap(f)(x)
    _traced(f, x)
    assert seen == [False, False]


@pytest.mark.parametrize("name", ["_tracing_state", "_functorch_level"])
def test_without_an_internal_of_torch(monkeypatch, name):
    """Another torch may not have it: then the Function runs."""
    monkeypatch.setattr(L, name, None)
    assert not L.plain_forward(torch.ones(2))


@pytest.mark.gpu
def test_unroute_add_without_an_addend(dev):
    from mintext_amd.kernels import unroute
    from mintext_amd.kernels.moe_dispatch import unroute_add

    x, w = torch.randn(8, 64, device=dev), torch.rand(4, 2, device=dev)
    si = torch.arange(8, device=dev, dtype=torch.int32)
    assert torch.equal(unroute_add(x, si, w, 2, None), unroute(x, si, w, 2))


@pytest.mark.gpu
@pytest.mark.parametrize("op", ["grouped_matmul", "route", "unroute"])
def test_traced_ops_compute(dev, op):
    """A trace made without gradients computes on new inputs."""
    from mintext_amd.kernels import grouped_matmul, route, unroute

    T, K, E, D = 24, 2, 4, 64
    idx = (torch.arange(T * K, device=dev, dtype=torch.int32) % E).reshape(T, K)
    gs = torch.full((E,), T * K // E, device=dev, dtype=torch.int32)
    w = torch.randn(E, D, D, device=dev).bfloat16()
    tw = torch.rand(T, K, device=dev)
    f, rows = {
        "grouped_matmul": (lambda x: grouped_matmul(x, w, gs), T * K),
        "route": (lambda x: route(x, idx, E)[0], T),
        "unroute": (lambda x: unroute(x, torch.arange(T * K, device=dev, dtype=torch.int32), tw, K), T * K),
    }[op]
    a, b = (torch.randn(rows, D, device=dev).bfloat16() for _ in range(2))
    traced = _traced(f, a)
    assert torch.equal(traced(b), f(b))
