"""Fused linear-LogP of a hidden size that whole 16-byte chunks do not divide: every token count runs the element-wise
loader, whichever grid it would take otherwise."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tokens", [40, 300, 385, 500, 1024, 1025])
def test_every_grid_reads_whole_rows_only(tokens):
    from rl_engine.ops.logprob import deterministic_linear_logp

    vocab, hidden = 1200, 100
    gen = torch.Generator(device="cuda").manual_seed(tokens)
    h = torch.randn((tokens, hidden), generator=gen, device="cuda", dtype=torch.bfloat16)
    w = torch.randn((vocab, hidden), generator=gen, device="cuda", dtype=torch.bfloat16).mul_(0.3)
    ids = torch.randint(0, vocab, (tokens,), generator=gen, device="cuda")
    logp, lse = deterministic_linear_logp(h, w, ids)
    z = h.double() @ w.double().t()
    want_lse = z.logsumexp(1)
    # fp32 sums of 100 products and of 1200 exponentials of logits below 20
    assert float((lse.double() - want_lse).abs().max()) < 2e-5
    assert float((logp.double() - (z.gather(1, ids[:, None])[:, 0] - want_lse)).abs().max()) < 2e-5
    few, few_lse = deterministic_linear_logp(h[:7], w, ids[:7])
    assert torch.equal(few.view(torch.int32), logp[:7].view(torch.int32)) and torch.equal(few_lse, lse[:7])
