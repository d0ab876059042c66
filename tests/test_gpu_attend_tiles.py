"""The attention of a chunk at the edges of its tiles: cluster runs and causal windows
whose lengths sit around multiples of the 32-key tile, work items with a full, a nearly
empty and a single-query last tile of queries, for every head grouping and both head
dimensions, on the whole grid and on one of 8 blocks (each block then works through
many items, in the two-block form, which dense chunks of this size take only with an
explicit grid; test_gpu_attend_forms.py has the launches that pick it by themselves).  Against
fp64 attention over the explicit key sets."""
from __future__ import annotations

import pytest
import torch

from gpu_util import assert_close_bf16

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _chunk_reference(q, k_rows, v_rows, keep):
    """fp64 attention of one KV head: q [Q, G, D], rows [N, D], keep [Q, N] bool."""
    s = torch.einsum("qgd,nd->qgn", q.double(), k_rows.double()) * q.shape[-1] ** -0.5
    p = torch.softmax(s.masked_fill(~keep[:, None], float("-inf")), dim=-1)
    return torch.einsum("qgn,nd->qgd", p, v_rows.double())


@pytest.mark.parametrize("hkv,g,d", [(1, 1, 128), (2, 2, 256), (1, 4, 256), (2, 4, 128), (1, 8, 256), (1, 8, 128)])
@pytest.mark.parametrize("qn,grid", [(1, None), (31, 8), (33, None), (200, 8)])
def test_sparse_chunk_at_tile_edges(hkv, g, d, qn, grid):
    from semblo_amd.kv_outer import kv_outer_attention
    gen = torch.Generator().manual_seed(1000 * d + 10 * g + qn)
    c = 32
    lens = torch.tensor([1, 31, 32, 33, 63, 64, 65, 96, 97, 0] + [16] * 22)
    visible = torch.stack([lens.roll(h) for h in range(hkv)])
    indptr = torch.zeros(hkv, c + 1, dtype=torch.int64)
    indptr[:, 1:] = ((visible + 15) // 16 * 16).cumsum(1)
    width = int(indptr[:, -1].max())
    packed = torch.randn(2, width, hkv, d, generator=gen).to(torch.bfloat16)
    q = torch.randn(qn, hkv * g, d, generator=gen).to(torch.bfloat16)
    kw, vw = (torch.randn(qn, hkv, d, generator=gen).to(torch.bfloat16) for _ in range(2))
    sel = torch.rand(qn, hkv, c, generator=gen) < 0.5
    words = (sel.view(qn, hkv, 1, 32).long() << torch.arange(32)).sum(-1)
    words = torch.where(words >= 2 ** 31, words - 2 ** 32, words).to(torch.int32)
    start = 5000
    out, _ = kv_outer_attention(q.to(DEV), packed.to(DEV), words.to(DEV), visible.int().to(DEV),
                                indptr.int().to(DEV), sm_scale=d ** -0.5,
                                local_kv=(kw.to(DEV), vw.to(DEV)), chunk_start=start, wstart=start, grid=grid)
    causal = torch.ones(qn, qn, dtype=torch.bool).tril()
    want = torch.empty(qn, hkv * g, d, dtype=torch.float64)
    for h in range(hkv):
        rows = torch.cat([torch.arange(int(indptr[h, i]), int(indptr[h, i] + visible[h, i])) for i in range(c)])
        owner = torch.repeat_interleave(torch.arange(c), visible[h])
        keep = torch.cat([sel[:, h][:, owner], causal], dim=1)
        want[:, h * g:(h + 1) * g] = _chunk_reference(
            q[:, h * g:(h + 1) * g], torch.cat([packed[0, rows, h], kw[:, h]]),
            torch.cat([packed[1, rows, h], vw[:, h]]), keep)
    assert_close_bf16(out.cpu(), want, f"sparse chunk hkv={hkv} g={g} d={d} qn={qn}")


@pytest.mark.parametrize("hkv,g,d", [(2, 4, 256), (1, 8, 128), (1, 1, 256)])
@pytest.mark.parametrize("start,qn,grid", [(0, 1, None), (31, 33, None), (64, 97, 8), (200, 129, None),
                                           (0, 65, -1), (200, 129, -1)])
@pytest.mark.parametrize("transposed,tower", [(False, False), (True, False), (False, True)])
def test_dense_chunk_at_tile_edges(hkv, g, d, start, qn, grid, transposed, tower):
    """Both kernel forms (the two-block one at grid 8, the other at these sizes and where grid -1
    asks for the one that leaves room), also with the output's
    heads outside its queries (a strided output) and with keys that tower over the first
    tile's (every 61st lies along the queries' common direction: the items are redone)."""
    from semblo_amd.kv_outer import dense_causal_attention
    gen = torch.Generator().manual_seed(d + g + start + qn)
    q = torch.randn(qn, hkv * g, d, generator=gen)
    k, v = (torch.randn(start + qn, hkv, d, generator=gen).to(torch.bfloat16) for _ in range(2))
    if tower:
        u = torch.randn(d, generator=gen)
        q = q + 3 * u
        k[40::61] = (3 * u).to(torch.bfloat16)
    q = q.to(torch.bfloat16)
    out = None
    if transposed:
        out = torch.empty(hkv * g, qn, d, dtype=torch.bfloat16, device=DEV).transpose(0, 1)
    got = dense_causal_attention(q.to(DEV), k.to(DEV), v.to(DEV), sm_scale=d ** -0.5, chunk_start=start,
                                 out=out, grid=grid)
    keep = torch.arange(start + qn)[None] <= (start + torch.arange(qn))[:, None]
    want = torch.cat([_chunk_reference(q[:, h * g:(h + 1) * g], k[:, h], v[:, h], keep) for h in range(hkv)], dim=1)
    assert_close_bf16(got.cpu(), want, f"dense chunk hkv={hkv} g={g} d={d} {start}+{qn}")
