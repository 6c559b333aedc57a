"""GPU parity of the one-workgroup route at its step of 1024 ids, its largest count and its largest number
of experts: whole numbers, equal to numpy's stable sort, invalid ids last and uncounted."""
from __future__ import annotations

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,K,E", [(1, 1, 40), (1, 8, 128), (127, 8, 64), (128, 8, 33), (129, 8, 256), (683, 3, 500),
                                   (256, 8, 960), (257, 8, 128), (40, 4, 1023)])
@pytest.mark.parametrize("invalid", [False, True])
def test_route_few_ids(dev, N, K, E, invalid):
    from mintext_amd.kernels.moe_dispatch import route_indices

    rng = np.random.default_rng(N * K + E)
    idx = rng.integers(0, E, (N, K)).astype(np.int32)
    if invalid:
        idx[rng.random((N, K)) < 0.1] = -1
        idx[rng.random((N, K)) < 0.1] = E + 3
    si, gs, inv = route_indices(torch.from_numpy(idx).to(dev), E)
    keys = np.where((idx < 0) | (idx >= E), E, idx).ravel()
    perm, counts = np.argsort(keys, kind="stable"), np.bincount(keys, minlength=E + 1)[:E]
    assert np.array_equal(si.cpu().numpy(), perm)
    assert np.array_equal(gs.cpu().numpy(), counts)
    assert np.array_equal(inv.cpu().numpy()[perm], np.arange(N * K))
