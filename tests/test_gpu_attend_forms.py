"""The attention's two kernel forms where the launch picks them by itself (no explicit grid):
a dense chunk with an item for every compute unit and one past that, sparse chunks on either
side of the lines, each block then working through several items, the last tiles ragged.
Against fp64 attention over the explicit key sets."""
from __future__ import annotations

import pytest
import torch

from gpu_util import assert_close_bf16

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _units():
    return torch.cuda.get_device_properties(0).multi_processor_count


def _attend(q, k, v, keep):
    """fp64 attention of one head on the GPU: q [Q, D], k and v [N, D], keep [Q, N] bool."""
    s = q.double() @ k.double().T * q.shape[-1] ** -0.5
    return torch.softmax(s.masked_fill(~keep, float("-inf")), dim=-1) @ v.double()


def _queries(items, hkv, g):
    """An odd number of queries that makes about this many window items."""
    return max(1, items // hkv * (128 // g) - 37 % (128 // g))


@pytest.mark.parametrize("hkv,g,d,share", [
    (2, 8, 256, 1.0), (2, 8, 256, 1.02), (4, 4, 256, 2.5), (16, 1, 256, 1.05),    # one block, then two
    (16, 2, 128, 1.2), (16, 2, 128, 1.3), (4, 8, 128, 2.1)])                       # one, two, one
def test_dense_chunk_past_an_item_per_unit(hkv, g, d, share):
    from semblo_amd.kv_outer import dense_causal_attention
    qn = _queries(int(share * _units()), hkv, g)
    gen = torch.Generator(device=DEV).manual_seed(qn + d)
    start = 45
    q = torch.randn(qn, hkv * g, d, generator=gen, device=DEV).to(torch.bfloat16)
    k, v = (torch.randn(start + qn, hkv, d, generator=gen, device=DEV).to(torch.bfloat16) for _ in range(2))
    got = dense_causal_attention(q, k, v, sm_scale=d ** -0.5, chunk_start=start)
    keep = torch.arange(start + qn, device=DEV)[None] <= (start + torch.arange(qn, device=DEV))[:, None]
    want = torch.stack([_attend(q[:, j], k[:, j // g], v[:, j // g], keep) for j in range(hkv * g)], dim=1)
    assert_close_bf16(got.cpu(), want.cpu(), f"dense hkv={hkv} g={g} d={d} qn={qn}")


# the form: one block where none is asked for by the items (or with grid -1), two from the line on
@pytest.mark.parametrize("hkv,g,d,share,start,grid,tower", [
    (2, 8, 256, 0.1, 10000, None, False), (2, 8, 256, 0.1, 10000, None, True),      # one block: long runs
    (2, 8, 256, 0.1, 5000, -1, True), (4, 4, 256, 0.2, 10000, None, True),
    (2, 8, 256, 0.1, 5000, None, True),                                             # two: short runs
    (4, 4, 256, 0.9, 10000, None, True), (2, 8, 256, 1.1, 10000, None, False),      # one, two: items
    (8, 2, 256, 0.9, 5000, None, False), (16, 2, 256, 1.1, 10000, None, False),     # one, two
    (16, 2, 128, 1.1, 5000, None, True), (16, 2, 128, 1.4, 5000, None, True),       # one, two
    (16, 1, 128, 1.4, 5000, None, False), (4, 8, 128, 1.4, 5000, None, True)])      # two, one
def test_sparse_chunk_on_both_sides_of_the_lines(hkv, g, d, share, start, grid, tower):
    """``tower``: keys that tower over a run's first tile (every 61st row lies along the queries'
    common direction: those items are run again with their rows' maxima)."""
    from semblo_amd.kv_outer import kv_outer_attention
    qn = _queries(int(share * _units()), hkv, g)
    gen = torch.Generator(device=DEV).manual_seed(qn + d + start)
    c = 32
    lens = torch.tensor([1, 31, 32, 33, 63, 64, 65, 96, 97, 0, 500] + [16] * 21)
    visible = torch.stack([lens.roll(h) for h in range(hkv)])
    indptr = torch.zeros(hkv, c + 1, dtype=torch.int64)
    indptr[:, 1:] = ((visible + 15) // 16 * 16).cumsum(1)
    packed = torch.randn(2, int(indptr[:, -1].max()), hkv, d, generator=gen, device=DEV)
    q = torch.randn(qn, hkv * g, d, generator=gen, device=DEV)
    if tower:
        u = torch.randn(d, generator=gen, device=DEV)
        q = q + 3 * u
        packed[0, 40::61] = 3 * u
    q, packed = q.to(torch.bfloat16), packed.to(torch.bfloat16)
    kw, vw = (torch.randn(qn, hkv, d, generator=gen, device=DEV).to(torch.bfloat16) for _ in range(2))
    sel = torch.rand(qn, hkv, c, generator=gen, device=DEV) < 0.4
    words = (sel.view(qn, hkv, 1, 32).long() << torch.arange(32, device=DEV)).sum(-1)
    words = torch.where(words >= 2 ** 31, words - 2 ** 32, words).to(torch.int32)
    out, _ = kv_outer_attention(q, packed, words, visible.int().to(DEV), indptr.int().to(DEV), sm_scale=d ** -0.5,
                                local_kv=(kw, vw), chunk_start=start, wstart=start, grid=grid)
    causal = torch.ones(qn, qn, dtype=torch.bool, device=DEV).tril()
    want = torch.empty(qn, hkv * g, d, dtype=torch.float64, device=DEV)
    for h in range(hkv):
        rows = torch.cat([torch.arange(int(indptr[h, i]), int(indptr[h, i] + visible[h, i])) for i in range(c)]).to(DEV)
        owner = torch.repeat_interleave(torch.arange(c), visible[h]).to(DEV)
        keep = torch.cat([sel[:, h][:, owner], causal], dim=1)
        k, v = torch.cat([packed[0, rows, h], kw[:, h]]), torch.cat([packed[1, rows, h], vw[:, h]])
        for j in range(h * g, (h + 1) * g):
            want[:, j] = _attend(q[:, j], k, v, keep)
    assert_close_bf16(out.cpu(), want.cpu(), f"sparse hkv={hkv} g={g} d={d} qn={qn} start={start}")
