"""Test configuration: the ``gpu`` marker and shared helpers.

CPU tests (``-m "not gpu"``) pin the oracle against the golden fixtures and check the C-ABI
library's exports and host-side argument validation.  GPU tests (``-m gpu``) compare the HIP
kernels, called through the C-ABI, with the oracle.
"""
from __future__ import annotations

import sys
from pathlib import Path

import numpy as np
import pytest

ROOT = Path(__file__).resolve().parents[1]
if str(ROOT) not in sys.path:
    sys.path.insert(0, str(ROOT))

GOLDEN = ROOT / "tests" / "golden"


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs a ROCm GPU (MI355X) and the built HIP library")


def golden(name: str):
    return np.load(GOLDEN / f"{name}.npz", allow_pickle=False)


@pytest.fixture(scope="session")
def dev():
    import torch

    if not torch.cuda.is_available():
        pytest.skip("no ROCm GPU visible")
    from mintext_amd import _lib

    _lib.lib()  # raises if the HIP library is missing: GPU tests never run without it
    return torch.device("cuda:0")


def rel_err(a, b) -> float:
    a = np.asarray(a, dtype=np.float64)
    b = np.asarray(b, dtype=np.float64)
    den = np.linalg.norm(b.ravel())
    return float(np.linalg.norm((a - b).ravel()) / (den if den > 0 else 1.0))


def tile_list_workspace_bytes(M: int, E: int) -> int:
    """The tile-list part of the grouped-GEMM workspace (mtx_gmm_workspace_size without the split
    tail): with it every tile runs whole, so any two kernels agree bit for bit."""
    up = lambda a, b: (a + b - 1) // b * b
    return up(up((48 + 2 * E + 1) * 4, 256) + (-(-M // 64) + E + 1) * 16, 256)


def split_pieces(m_tiles: int, n_tiles: int, stages: int, few_stages: int, cus: int = 32) -> int:
    """Pieces of the split-tail tiles of a launch of 256-row tiles (XCDs with a full share of them): the rule
    of ``split_pieces`` in gmm.hip, few_stages 16 in the 8-wave kernel and 32 in the one-wave-per-SIMD one."""
    tiles = -(-m_tiles * n_tiles // 8)
    rem = tiles % cus
    if not 0 < rem <= 16 or 2 * rem > cus or stages < 40:
        return 1
    return min(4, cus // rem, max(stages // (few_stages if tiles <= 8 else 40), 1))


def launched(f) -> str:
    """The names of the kernels that ``f`` launches, one a line."""
    import torch
    from torch.profiler import ProfilerActivity, profile

    torch.cuda.synchronize()
    with profile(activities=[ProfilerActivity.CPU, ProfilerActivity.CUDA]) as p:
        f()
        torch.cuda.synchronize()
    return "\n".join(e.name for e in p.events() if e.device_type == torch.autograd.DeviceType.CUDA)
