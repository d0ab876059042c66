"""The selection kernel's forms against the oracle: cluster counts that fill a lane's share
and ones that do not, every head grouping (the softmax in the query's wave, or through the
table), budgets that nothing, one cluster, some and all clusters meet, odd and short
bisections, and scores far apart (the bisection ends early) or equal (it cannot)."""
from __future__ import annotations

import pytest
import torch

from gpu_util import compare_selection
from oracle import reference_cpu as ref

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("c,g,d,q", [(64, 1, 128, 5), (128, 2, 256, 37), (192, 4, 128, 33), (256, 4, 256, 9),
                                     (320, 8, 128, 17), (512, 1, 64, 6), (1024, 4, 256, 5), (128, 16, 128, 3)])
@pytest.mark.parametrize("kind,tau,iters", [("mixed", 0.1, 16), ("apart", 0.02, 16), ("equal", 0.1, 16),
                                            ("mixed", 0.1, 15), ("mixed", 0.1, 3)])
def test_selection_forms_match_the_oracle(c, g, d, q, kind, tau, iters):
    from semblo_amd.fused_select import theta_select_bitmask_flat
    gen = torch.Generator().manual_seed(c + 7 * g + d + iters)
    hkv = 2
    unit = torch.nn.functional.normalize
    cent = unit(torch.randn(hkv, c, d, generator=gen), dim=-1)
    if kind == "equal":
        cent[:, 1::2] = cent[:, ::2]                    # pairs of equal scores
    codebooks = cent.view(hkv, c, 2, d // 2).transpose(1, 2).to(torch.bfloat16).contiguous()
    vec = unit(torch.randn(q, hkv * g, d, generator=gen), dim=-1).to(torch.bfloat16)
    sizes = torch.randint(0, 200, (1, hkv, c), generator=gen, dtype=torch.int32)
    if kind == "equal":
        sizes[..., 1::2] = sizes[..., ::2]
    total = int(sizes.sum(-1).min())
    for target in (1, total // 16, total // 2, total, 2 * total):
        prob = torch.empty(q, hkv, c, device=DEV)
        theta = torch.empty(q, hkv, device=DEV)
        qmask = torch.empty(q, hkv, c // 32, dtype=torch.int32, device=DEV)
        counts, tokens = theta_select_bitmask_flat(
            vec.to(DEV)[:, :, None], None, codebooks.to(DEV), sizes.to(DEV), None, temperature=tau, beta=0.25,
            target_tokens=target, g_union=q, iters=iters, qmask=qmask, prob_out=prob, theta_out=theta)
        want_prob = ref.mixture_probs(vec, None, codebooks, tau)
        # fp32 sums in another order, base-2 hardware exp and log: about 1e-6 relative
        assert torch.allclose(prob.cpu(), want_prob, rtol=2e-5, atol=1e-9)
        want = ref.theta_select(prob.cpu(), sizes, beta=0.25, target_tokens=target, g_union=q, iters=iters)
        sel = ref.unpack_bits(qmask.cpu(), c)
        compare_selection(sel, want["sel"], want["score"], want["theta"], theta.cpu())
        assert torch.equal(counts.cpu(), sel.sum(-1).int())
        assert torch.equal(tokens.cpu(), (sel * sizes).sum(-1).int())
