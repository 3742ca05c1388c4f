"""Test configuration: the ``gpu`` marker and shared helpers."""

from __future__ import annotations

import contextlib
import sys
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
if str(ROOT) not in sys.path:
    sys.path.insert(0, str(ROOT))


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (runs through the HIP C-ABI library)")


def pytest_collection_modifyitems(config, items):
    import torch

    if torch.cuda.is_available():
        return
    skip = pytest.mark.skip(reason="no GPU in this environment")
    for item in items:
        if "gpu" in item.keywords:
            item.add_marker(skip)


@contextlib.contextmanager
def device_memory_left(nbytes: int):
    """Torch's allocator has ``nbytes`` of device memory to give and no more
    (its own limit, whatever the card still has; blocks under 1 MiB apart)."""

    import torch

    total = torch.cuda.get_device_properties(0).total_memory
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    taken = []
    try:
        torch.cuda.set_per_process_memory_fraction(torch.cuda.memory_reserved() / total)
        size = 1 << 30
        while size >= 1 << 20:  # what segments still in use have free
            try:
                taken.append(torch.empty(size, dtype=torch.uint8, device="cuda"))
            except torch.OutOfMemoryError:
                size //= 2
        torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + nbytes) / total)
        yield
        torch.cuda.synchronize()
    finally:
        del taken
        torch.cuda.set_per_process_memory_fraction(1.0)
