"""The plans of several sparse chunks in one call (sbsa_plan_chunks) against the plan of each
chunk: the same selections, sizes, reverse index and work list, whole numbers all, with a
ragged last chunk, a single chunk, and a capped partial buffer that some chunks pass."""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("length,hkv,g,d,step,first,cap_mb", [
    (4096, 2, 4, 128, 512, 1024, None), (3001, 4, 4, 256, 700, 1400, None), (2500, 1, 8, 128, 1024, 1024, None),
    (2049, 2, 1, 256, 1024, 1024, None), (4000, 2, 2, 128, 640, 1280, "3")])
def test_group_plan_equals_each_chunks_plan(length, hkv, g, d, step, first, cap_mb, monkeypatch):
    from semblo_amd.fused_prefill import CausalSnapshot, fused_chunk_plan, fused_chunks_plan
    from semblo_amd.kv_outer import PartialsGuard
    from semblo_amd.model import SembloQueryState
    from semblo_amd.state import ProductPostingIndex
    from semblo_amd.synthetic import mixture_layer
    from semblo_amd.trivial_router import trivial_router_vectors
    if cap_mb is not None:
        monkeypatch.setenv("SEMBLO_KV_OUTER_PARTIALS_CAP_MB", cap_mb)
    inp = mixture_layer(length, hkv * g, hkv, d, mixtures=64, seed=length + d, device=DEV)
    index = ProductPostingIndex.build(inp.k, torch.arange(length, device=DEV), router_pass=True)
    sel = dict(temperature=0.1, beta=0.25, target_tokens=length // 16, iters=16, keep_theta=True)
    group = fused_chunks_plan(inp.q[first:], index, first, step, guard=PartialsGuard(), **sel)
    snapshot = CausalSnapshot(index)
    starts = list(range(first, length, step))
    assert len(group) == len(starts)
    for pl, st in zip(group, starts):
        en = min(length, st + step)
        q = inp.q[st:en]
        vec = trivial_router_vectors(q, 1)
        state = SembloQueryState(vec[None, :, :, None], torch.ones(1, en - st, hkv * g, 1, device=DEV))
        # one chunk's own plan starts its window where the chunk does (past the dense prefix)
        one = fused_chunk_plan(q, state, index, snapshot, st, en - 1, dense_prefix_x=0, **sel)
        one.kv.prepare_work(q, hkv, index.bucket_indptr, PartialsGuard())
        assert (pl.chunk_start, pl.chunk_end, pl.wstart) == (one.chunk_start, one.chunk_end, one.wstart)
        assert torch.equal(pl.causal_sizes, one.causal_sizes) and torch.equal(pl.tokens, one.tokens)
        assert torch.equal(pl.theta, one.theta)
        a, b = pl.kv, one.kv
        nnz = int(b.nnz_d)
        assert int(a.nnz_d) == nnz and torch.equal(a.qmask, b.qmask) and torch.equal(a.counts, b.counts)
        assert torch.equal(a.rev_indptr, b.rev_indptr) and torch.equal(a.qvals[:nnz], b.qvals[:nnz])
        picked = ((b.qmask[..., None] >> torch.arange(32, device=DEV)) & 1).bool().flatten(2) & (b.nvis > 0)
        assert torch.equal(a.qrank[picked], b.qrank[picked])
        assert a.work[:2] == b.work[:2]
        assert torch.equal(a.work[3][:25], b.work[3][:25])           # segments, offsets, counters, overflow
        n_items = int(b.work[3][:8].sum())
        assert torch.equal(a.work[2][:n_items], b.work[2][:n_items])
        assert (a.work[4] is None) == (b.work[4] is None)
        if a.work[4] is not None:
            for w in (a.work, b.work):
                w[4][0].synchronize()
            assert int(a.work[4][1][0]) == int(b.work[4][1][0])
