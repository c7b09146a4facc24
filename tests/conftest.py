"""Shared fixtures.  GPU tests are marked `gpu`; everything else runs on the CPU."""

from __future__ import annotations

import sys
from pathlib import Path

import pytest

REPO = Path(__file__).resolve().parents[1]
if str(REPO) not in sys.path:
    sys.path.insert(0, str(REPO))

GOLDEN = REPO / "tests" / "golden"


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs a ROCm GPU (MI355X) and the built extension")


@pytest.fixture(scope="session")
def ref():
    from oracle.ref import RefEngine

    return RefEngine()


@pytest.fixture(scope="session")
def ext():
    import torch

    if not torch.cuda.is_available():
        pytest.fail("gpu test selected but no GPU is visible")
    from cugo_amd import load_extension

    return load_extension()


def announce(name: str) -> None:
    print(f"[case] {name}", flush=True)


def poison_free_memory() -> None:
    """Fills the GPU memory that torch's allocator hands out next with 0xA5 bytes, so that an
    element that a kernel does not write differs from what an earlier call left there."""
    import torch

    torch.cuda.empty_cache()
    held = [torch.full((2 << 30,), 0xA5, dtype=torch.uint8, device="cuda")]
    for k in range(9, 21):  # the allocator keeps sizes up to 1 MiB apart, in pieces
        held += [torch.full((1 << k,), 0xA5, dtype=torch.uint8, device="cuda") for _ in range(32)]
    del held
    assert bool((torch.empty(1 << 24, dtype=torch.uint8, device="cuda") == 0xA5).all())
