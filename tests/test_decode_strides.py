"""The decode step reads the new token's K and V rows with one row stride: rows laid out
differently are refused on the host, before any pointer is taken."""
from __future__ import annotations

from types import SimpleNamespace

import pytest
import torch


@pytest.mark.parametrize("odd", ["k rows", "v rows", "k inner", "v inner"])
def test_new_rows_of_another_layout_are_refused(odd):
    from semblo_amd.fused_decode import fused_decode_step
    hq, hkv, d = 8, 4, 64
    layer = SimpleNamespace(num_heads=hq, num_kv_heads=hkv, head_dim=d)
    arena = SimpleNamespace(num_clusters=64, suffix_splits=2)
    kv = {"k": torch.zeros(1, hkv, 1, d), "v": torch.zeros(1, hkv, 1, d)}
    which, what = odd.split()
    if what == "rows":
        kv[which] = torch.zeros(1, hkv, 8, d)[:, :, 3:4]             # a row of a longer block
    else:
        kv[which] = torch.zeros(d, hkv).t()[None, :, None]
    q = torch.zeros(1, hq, d)
    with pytest.raises(ValueError, match="one row stride"):
        fused_decode_step(layer, arena, q_post=q, q_pre=q, positions=torch.zeros(1, dtype=torch.int32),
                          k_post=kv["k"], v_states=kv["v"], output=torch.zeros(1, hq * d), temperature=0.1,
                          beta=0.25, target_tokens=64, sm_scale=0.1, num_splits=4, no_alloc=True)
