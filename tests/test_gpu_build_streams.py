"""The streams the layers' indexes are built on: one for all layers that a thread calls on one
stream, others for other streams and threads; the outputs do not depend on it."""
from __future__ import annotations

import threading

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def test_layers_on_different_streams_build_on_different_streams():
    from semblo_amd import model
    from semblo_amd.config import SembloRuntimeConfig
    from semblo_amd.synthetic import mixture_layer
    length, hq, hkv, d = 4000, 8, 2, 128
    cfg = SembloRuntimeConfig(num_q_heads=hq, num_kv_heads=hkv, head_dim=d, query_chunk_size=1000)
    inp = mixture_layer(length, hq, hkv, d, mixtures=16, seed=2)
    q, k, v = inp.q.to(DEV), inp.k.to(DEV), inp.v.to(DEV)
    layers = [model.SembloAttention(cfg, layer_name=f"stream.{i}") for i in range(4)]
    mains = [torch.cuda.Stream(), torch.cuda.Stream()]
    outs = [torch.empty(length, hq * d, dtype=torch.bfloat16, device=DEV) for _ in layers]
    used = []
    for i, layer in enumerate(layers):
        main = mains[i % 2]
        main.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(main):
            layer.prefill(q, q, k, k, v, outs[i])
            used.append(layer._build_stream(main))
    torch.cuda.synchronize()
    assert used[0] == used[2] and used[1] == used[3] and used[0] != used[1]
    assert not set(used) & set(mains)
    other = []
    t = threading.Thread(target=lambda: other.append(layers[0]._build_stream(mains[0])))
    t.start()
    t.join()
    assert other[0] != used[0]
    for out in outs[1:]:
        assert torch.equal(out, outs[0])
