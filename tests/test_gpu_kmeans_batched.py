"""The batched index build (every KV head's fit in one call, sbsa_kmeans_fit) against the
build head after head, which the other tests check against the oracle and the reference's
golden vectors: the same index bit for bit, whatever restarts the heads take, and a build
that needs more restarts than are drawn ahead falls back to the sequential one."""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _keys(length, hkv, d, mixtures, seed):
    """Mixture keys; few mixtures leave clusters empty, a different number in every head."""
    gen = torch.Generator().manual_seed(seed)
    out = torch.empty(length, hkv, d)
    for h in range(hkv):
        m = max(1, mixtures >> h)
        centres = torch.randn(m, d, generator=gen)
        out[:, h] = centres[torch.randint(0, m, (length,), generator=gen)]
        out[:, h] += 0.3 * torch.randn(length, d, generator=gen)
    return out.to(torch.bfloat16).to(DEV)


def _fields(index):
    return (index.codebooks, index.posting_positions, index.bucket_indptr, index.bucket_sizes,
            index.inverse_positions())


@pytest.mark.parametrize("length,hkv,d,mixtures", [
    (1000, 1, 128, 64), (2051, 2, 256, 300), (4096, 4, 64, 200), (9001, 4, 128, 2000), (5000, 8, 128, 512),
    (3000, 4, 256, 16)])
@pytest.mark.parametrize("seed", [0, 5])
def test_batched_build_equals_the_sequential_one(length, hkv, d, mixtures, seed, monkeypatch):
    from semblo_amd import state
    keys = _keys(length, hkv, d, mixtures, seed + length)
    positions = torch.arange(length, device=DEV)
    batched = []
    real = state._fit_batched
    monkeypatch.setattr(state, "_fit_batched", lambda *a, **kw: batched.append(real(*a, **kw)) or batched[-1])
    got = state.ProductPostingIndex.build(keys, positions, codebook_seed=seed, router_pass=True)
    monkeypatch.setattr(state, "_fit_batched", lambda *a, **kw: None)
    want = state.ProductPostingIndex.build(keys, positions, codebook_seed=seed, router_pass=True)
    assert len(batched) == 1
    for a, b in zip(_fields(got), _fields(want)):
        assert a.shape == b.shape and torch.equal(a, b)
    print("batched" if batched[0] is not None else "fell back")


def test_batched_build_reads_strided_keys():
    """Keys as a view of a fused projection's rows (strides past the heads)."""
    from semblo_amd import state
    keys = _keys(2000, 2, 128, 100, 3)
    fused = torch.zeros(2000, 4, 128, dtype=torch.bfloat16, device=DEV)
    fused[:, 1:3] = keys
    positions = torch.arange(2000, device=DEV)
    a = state.ProductPostingIndex.build(keys, positions, router_pass=True)
    b = state.ProductPostingIndex.build(fused[:, 1:3], positions, router_pass=True)
    for x, y in zip(_fields(a), _fields(b)):
        assert torch.equal(x, y)
