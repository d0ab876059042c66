"""The batched build's random draws (sbsa_kmeans_draws, a host function) against the draws
the reference makes with torch's CPU generator: head after head a permutation of the keys,
one of the sample, and one of the sample per restart.  CPU only."""
from __future__ import annotations

import pytest
import torch


@pytest.mark.parametrize("seed,length,fit_n,heads,c,ahead", [
    (0, 200, 200, 1, 64, 2), (7, 1000, 400, 3, 64, 2), (123456789, 5003, 4096, 2, 128, 2),
    (2 ** 31 + 5, 8193, 8192, 4, 128, 2), (2 ** 40 + 3, 777, 128, 2, 128, 1), (3, 64, 64, 2, 64, 3)])
def test_draws_equal_torch_randperm(seed, length, fit_n, heads, c, ahead):
    from semblo_amd import _lib
    if not _lib.LIB_PATH.exists():
        pytest.skip("libsbsa.so is not built here")
    n = _lib.query("sbsa_kmeans_draw_ints", fit_n, heads, c, ahead)
    out = torch.empty(n, dtype=torch.int32)
    scratch = torch.empty(_lib.query("sbsa_kmeans_draw_scratch_ints", length, fit_n, heads, ahead), dtype=torch.int32)
    _lib.call("sbsa_kmeans_draws", seed & 0xffffffff, length, fit_n, heads, c, ahead, out.data_ptr(),
              scratch.data_ptr())
    fits = heads + ahead * (heads * (heads - 1) // 2)
    size = fit_n + (1 + ahead) * c
    assert n == fits * (size + 1)
    sets, head_of = out[:fits * size].view(fits, size), out[fits * size:]
    fit = 0
    for h in range(heads):
        for restarts in range(ahead * h + 1):
            gen = torch.Generator().manual_seed(seed)
            for _ in range(h):                       # the earlier heads, `restarts` spread over them
                torch.randperm(length, generator=gen)
                torch.randperm(fit_n, generator=gen)
            for _ in range(restarts):
                torch.randperm(fit_n, generator=gen)
            want = [torch.randperm(length, generator=gen)[:fit_n], torch.randperm(fit_n, generator=gen)[:c]]
            want += [torch.randperm(fit_n, generator=gen)[:c] for _ in range(ahead)]
            assert torch.equal(sets[fit].long(), torch.cat(want)), (h, restarts)
            assert int(head_of[fit]) == h
            fit += 1
    assert fit == fits


def test_draws_refuse_bad_shapes():
    from semblo_amd import _lib
    if not _lib.LIB_PATH.exists():
        pytest.skip("libsbsa.so is not built here")
    lib = _lib.load()
    out = torch.empty(100000, dtype=torch.int32)
    assert lib.sbsa_kmeans_draws(1, 100, 200, 1, 64, 2, out.data_ptr(), out.data_ptr()) == 1      # sample larger than the keys
    assert lib.sbsa_kmeans_draws(1, 200, 32, 1, 64, 2, out.data_ptr(), out.data_ptr()) == 1       # fewer rows than clusters
    assert lib.sbsa_kmeans_draws(1, 200, 100, 1, 64, 2, None, out.data_ptr()) == 1


@pytest.mark.parametrize("seed,length,fit_n,before,restarts,heads,c,ahead", [
    (0, 200, 200, 0, 0, 1, 64, 8), (7, 1000, 400, 1, 3, 1, 64, 8), (5, 5003, 4096, 2, 9, 2, 128, 2),
    (2 ** 31 + 5, 8193, 8192, 3, 20, 1, 128, 8), (11, 64, 64, 1, 0, 2, 64, 2), (4, 313, 313, 1, 0, 1, 64, 2)])
def test_draws_after_earlier_heads_and_restarts(seed, length, fit_n, before, restarts, heads, c, ahead):
    """The draws from where earlier heads and their restarts left the generator (the last case: 624
    words before, a whole block)."""
    from semblo_amd import _lib
    if not _lib.LIB_PATH.exists():
        pytest.skip("libsbsa.so is not built here")
    out = torch.empty(_lib.query("sbsa_kmeans_draw_ints", fit_n, heads, c, ahead), dtype=torch.int32)
    scratch = torch.empty(_lib.query("sbsa_kmeans_draw_scratch_ints", length, fit_n, heads, ahead), dtype=torch.int32)
    _lib.call("sbsa_kmeans_draws_after", seed & 0xffffffff, before, restarts, length, fit_n, heads, c, ahead,
              out.data_ptr(), scratch.data_ptr())
    gen = torch.Generator().manual_seed(seed)
    for _ in range(before):
        torch.randperm(length, generator=gen)
        torch.randperm(fit_n, generator=gen)
    for _ in range(restarts):
        torch.randperm(fit_n, generator=gen)
    size = fit_n + (1 + ahead) * c
    fit = 0
    for h in range(heads):
        state = gen.get_state()
        for r in range(ahead * h + 1):
            gen.set_state(state)
            for _ in range(r):
                torch.randperm(fit_n, generator=gen)
            want = [torch.randperm(length, generator=gen)[:fit_n], torch.randperm(fit_n, generator=gen)[:c]]
            want += [torch.randperm(fit_n, generator=gen)[:c] for _ in range(ahead)]
            assert torch.equal(out[fit * size:(fit + 1) * size].long(), torch.cat(want)), (h, r)
            fit += 1
        gen.set_state(state)
        torch.randperm(length, generator=gen)
        torch.randperm(fit_n, generator=gen)
