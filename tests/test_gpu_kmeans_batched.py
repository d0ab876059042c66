"""The batched index build (every KV head's fit in one call, sbsa_kmeans_fit) against the
build head after head, which the other tests check against the oracle and the reference's
golden vectors: the same index bit for bit, whatever restarts the heads take.  A head that
needs more restarts than are drawn ahead is fitted again alone, and so are those after it until
one needs no more; only past the restarts that one call can draw is the build the sequential one."""
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
    assert len(batched) == 1 and batched[0] is not None
    for a, b in zip(_fields(got), _fields(want)):
        assert a.shape == b.shape and torch.equal(a, b)


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


@pytest.mark.parametrize("length,hkv,d,repeated,iters,calls", [
    (3000, 1, 128, (0,), 8, [1, 1]), (3000, 5, 64, (1,), 8, [5, 1, 1, 2]),
    (5003, 4, 256, (0, 1, 2, 3), 8, [4, 1, 1, 1, 1]), (3000, 4, 64, (0, 3), 8, [4, 1, 1, 2, 1]),
    (2500, 3, 128, (2,), 5, [3, 1]), (2500, 2, 128, (0,), 2, [2]), (2500, 2, 128, (1,), 12, [2, 1])])
def test_heads_that_restart_more_than_is_drawn_ahead(length, hkv, d, repeated, iters, calls, monkeypatch):
    """Heads of 70 distinct keys leave some of 128 clusters empty in every iteration (past 8 iterations
    that is more than one call draws: the sequential build)."""
    from semblo_amd import _lib, state
    keys = _keys(length, hkv, d, 4000, length)
    for h in repeated:
        keys[:, h] = keys[:70, h].repeat(-(-length // 70), 1)[:length]
    positions = torch.arange(length, device=DEV)
    heads, real = [], _lib.call

    def call(name, *a):
        if name == "sbsa_kmeans_fit_counted":
            heads.append(a[4])
        return real(name, *a)
    monkeypatch.setattr(_lib, "call", call)
    got = state.ProductPostingIndex.build(keys, positions, codebook_seed=2, router_pass=True, fit_iters=iters)
    monkeypatch.setattr(_lib, "call", real)
    assert heads == calls
    monkeypatch.setattr(state, "_fit_batched", lambda *a, **kw: None)
    want = state.ProductPostingIndex.build(keys, positions, codebook_seed=2, router_pass=True, fit_iters=iters)
    for a, b in zip(_fields(got), _fields(want)):
        assert a.shape == b.shape and torch.equal(a, b)
