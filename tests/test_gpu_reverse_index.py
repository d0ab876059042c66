"""The reverse index in segments against the form without scratch: the same lists, counts,
starts and ranks, whole numbers all, at the segments' edges and with dead clusters."""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("qn", [1, 63, 255, 256, 257, 1000])
@pytest.mark.parametrize("hkv,c,share", [(1, 64, 0.3), (4, 128, 0.2), (2, 1024, 0.05), (3, 96, 1.0), (2, 32, 0.0)])
def test_segments_equal_one_block_per_cluster(qn, hkv, c, share):
    from semblo_amd import _lib
    gen = torch.Generator().manual_seed(qn * 7 + c)
    sel = torch.rand(qn, hkv, c, generator=gen) < share
    words = (sel.view(qn, hkv, c // 32, 32).long() << torch.arange(32)).sum(-1)
    qmask = torch.where(words >= 2 ** 31, words - 2 ** 32, words).to(torch.int32).to(DEV)
    live = (torch.rand(hkv, c, generator=gen) < 0.9).to(torch.int32).to(DEV)
    got = []
    for cap in (qn * hkv * c, _lib.query("sbsa_reverse_index_ints", qn, hkv, c)):
        counts = torch.empty(hkv, c, dtype=torch.int32, device=DEV)
        indptr = torch.empty(hkv * c + 1, dtype=torch.int32, device=DEV)
        nnz = torch.empty(1, dtype=torch.int64, device=DEV)
        qvals = torch.empty(cap, dtype=torch.int32, device=DEV)
        qrank = torch.full((qn, hkv, c), -1, dtype=torch.int32, device=DEV)
        _lib.call("sbsa_reverse_index", _lib.ptr(qmask), qn, hkv, c, _lib.ptr(live), _lib.ptr(counts),
                  _lib.ptr(indptr), _lib.ptr(nnz), _lib.ptr(qvals), cap, _lib.ptr(qrank), _lib.stream())
        got.append((counts, indptr, nnz, qvals[:int(nnz)], qrank))
    for a, b in zip(*got):
        assert torch.equal(a, b)
    assert int(got[0][2]) == int((sel.to(DEV) & (live > 0)).sum())
