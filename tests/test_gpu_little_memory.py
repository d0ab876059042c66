"""The index build and the layer's plans where memory is short: every head's fit at once, or the
plans of several chunks in one call, need more than head after head and chunk after chunk, and
give way to them with the same results."""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def test_build_head_after_head_where_all_at_once_does_not_fit(limit_memory):
    """Four key spaces of 65536 x 256 take 403 MB in one call, one 101 MB."""
    from semblo_amd import state
    gen = torch.Generator(device=DEV).manual_seed(1)
    keys = torch.randn(65536, 4, 256, generator=gen, device=DEV).to(torch.bfloat16)
    positions = torch.arange(65536, device=DEV)

    def build():
        x = state.ProductPostingIndex.build(keys, positions, codebook_seed=3, router_pass=True)
        return (x.codebooks, x.posting_positions, x.bucket_indptr, x.bucket_sizes, x.inverse_positions())
    want = build()
    limit_memory(250 << 20)
    for a, b in zip(build(), want):
        assert torch.equal(a, b)


def test_plans_chunk_after_chunk_where_a_group_does_not_fit(monkeypatch):
    from semblo_amd import model
    from semblo_amd.config import SembloRuntimeConfig
    from semblo_amd.synthetic import mixture_layer
    length, hq, hkv, d = 6000, 8, 2, 128
    inp = mixture_layer(length, hq, hkv, d, mixtures=16, seed=2)
    q, k, v = inp.q.to(DEV), inp.k.to(DEV), inp.v.to(DEV)
    outs = []

    def no_room(*a, **kw):
        raise torch.OutOfMemoryError("no room")
    for plan in (model.fused_chunks_plan, no_room):
        monkeypatch.setattr(model, "fused_chunks_plan", plan)
        layer = model.SembloAttention(SembloRuntimeConfig(num_q_heads=hq, num_kv_heads=hkv, head_dim=d,
                                                          query_chunk_size=1000), layer_name=f"room.{len(outs)}")
        out = torch.empty(length, hq * d, dtype=torch.bfloat16, device=DEV)
        outs.append(layer.prefill(q, q, k, k, v, out))
    assert torch.equal(*outs)
