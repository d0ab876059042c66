"""kv_outer_attention's partial count and partial rows: the count comes without a copy in the
stream between the reverse index and the attention, on a stream of its own too, and a GPU
without room for the rows' bound takes them at the exact count."""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _chunk(qn, hkv, g, d, c, share, seed=0):
    gen = torch.Generator(device=DEV).manual_seed(seed)

    def normal(*shape):
        return torch.randn(*shape, generator=gen, device=DEV).to(torch.bfloat16)
    visible = torch.randint(0, 40, (hkv, c), generator=gen, device=DEV)
    indptr = torch.zeros(hkv, c + 1, dtype=torch.int64, device=DEV)
    indptr[:, 1:] = ((visible + 15) // 16 * 16).cumsum(1)
    sel = torch.rand(qn, hkv, c, generator=gen, device=DEV) < share
    words = (sel.view(qn, hkv, c // 32, 32).long() << torch.arange(32, device=DEV)).sum(-1)
    words = torch.where(words >= 2 ** 31, words - 2 ** 32, words).to(torch.int32)
    start = 64 * c
    args = (normal(qn, hkv * g, d), normal(2, int(indptr[:, -1].max()), hkv, d), words, visible.int(), indptr.int())
    kw = dict(sm_scale=d ** -0.5, local_kv=(normal(qn, hkv, d), normal(qn, hkv, d)), chunk_start=start, wstart=start)
    return args, kw, int((sel & (visible > 0)).sum())


@pytest.mark.parametrize("qn,hkv,g,d,c", [(1, 1, 8, 128, 32), (300, 4, 4, 256, 128), (5000, 2, 2, 128, 64)])
@pytest.mark.parametrize("own_stream", [False, True])
def test_the_count_comes_without_a_copy(qn, hkv, g, d, c, own_stream, monkeypatch):
    from semblo_amd.kv_outer import kv_outer_attention
    args, kw, want = _chunk(qn, hkv, g, d, c, 0.2, seed=qn)
    ref = kv_outer_attention(*args, **kw)[0]
    copies = []
    real = torch.Tensor.copy_
    monkeypatch.setattr(torch.Tensor, "copy_", lambda t, *a, **k: copies.append(t.shape) or real(t, *a, **k))
    stream = torch.cuda.Stream() if own_stream else torch.cuda.current_stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        for _ in range(3):
            out, stats = kv_outer_attention(*args, **kw)
            assert stats["partials"] == want
    stream.synchronize()
    assert copies == [] and torch.equal(out, ref)


def test_rows_at_the_exact_count_where_the_bound_does_not_fit(limit_memory):
    """The bound of 4096 queries and 512 (head, cluster) takes 2.2 GB of rows, a twentieth of them
    selected 0.1 GB."""
    from semblo_amd.kv_outer import kv_outer_attention
    args, kw, want = _chunk(4096, 4, 4, 128, 128, 0.05)
    ref = kv_outer_attention(*args, **kw)[0]
    limit_memory(600 << 20)
    with pytest.raises(torch.OutOfMemoryError):
        torch.empty(2 << 30, dtype=torch.uint8, device=DEV)
    out, stats = kv_outer_attention(*args, **kw)
    assert stats["partials"] == want and torch.equal(out, ref)
