"""A repack hands the store's old rows over as a copy whose rows lie side by side, also for
one KV head, where the copy of a slice keeps the slice's row stride: the library would take
the longer range that stride spans for the old rows and refuse what overlaps it."""
from __future__ import annotations

from types import SimpleNamespace

import pytest
import torch


@pytest.mark.parametrize("hkv", [1, 2, 4])
def test_repack_passes_the_copys_own_row_length(hkv, monkeypatch):
    from semblo_amd import _lib, token_outer_prefill as top
    calls = []
    monkeypatch.setattr(_lib, "call", lambda name, *a: calls.append((name, a)))
    monkeypatch.setattr(_lib, "ptr", lambda t: t.data_ptr())
    monkeypatch.setattr(_lib, "stream", lambda device=None: 0)
    zeros = torch.zeros
    monkeypatch.setattr(torch, "zeros", lambda *a, pin_memory=False, **k: zeros(*a, **k))
    n, length, c, d = 20, 64, 2, 8
    s = object.__new__(top.TokenOuterPrefillSession)
    s._spare, s.repacks = None, 0
    s.verbose = False
    s._set_reserve = lambda reserve, device: None
    s.index = SimpleNamespace(packed_kv=zeros(2, length, hkv, d), num_buckets=c, extras={},
                              _inverse_positions=zeros(hkv, length, dtype=torch.int32),
                              posting_positions=zeros(hkv, length, dtype=torch.int32),
                              bucket_indptr=zeros(hkv, c + 1, dtype=torch.int32))
    s._repack(n, zeros(hkv, c, dtype=torch.int64))
    (name, args), = [x for x in calls if x[0] == "sbsa_repack_runs"]
    assert args[5] == n and args[7] == n
