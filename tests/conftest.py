"""Test configuration: the ``gpu`` marker and import paths."""
from __future__ import annotations

import sys
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
PKG_DIR = ROOT / "semantic-block-sparse-attention_amd"
for p in (str(ROOT), str(PKG_DIR), str(ROOT / "tests" / "golden")):
    if p not in sys.path:
        sys.path.insert(0, p)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (runs the HIP kernels)")
    config.addinivalue_line("markers", "emu: runs the HIP kernels on the CPU through tests/emu (slow)")


@pytest.fixture
def limit_memory():
    """Leaves torch's GPU allocator ``extra`` bytes past what is in use (a limit of the allocator)."""
    import torch

    def limit(extra):
        torch.cuda.synchronize()
        torch.cuda.empty_cache()
        total = torch.cuda.get_device_properties(0).total_memory
        torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + extra) / total)
    yield limit
    torch.cuda.set_per_process_memory_fraction(1.0)
