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
def limit_memory(monkeypatch):
    """Lets torch.empty refuse GPU memory past a size, as the allocator does where it is short."""
    import torch
    real = torch.empty

    def limit(most):
        def empty(*size, **kw):
            t = real(*size, **{**kw, "device": "meta", "pin_memory": False})
            if torch.device(kw.get("device") or "cpu").type == "cuda" and t.numel() * t.element_size() > most:
                raise torch.OutOfMemoryError("no room")
            return real(*size, **kw)
        monkeypatch.setattr(torch, "empty", empty)
    return limit
