"""Fused linear-LogP above 1024 tokens: a last token tile with few tokens runs as a smaller one, and the groups of token
tiles are of even width; the bits of every row are those of a call with that row and few others."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


# tokens: the last tile with 1, 64, 65, 128, 129 and 256 of them; one group of 5 to 11 tiles, two (8 + 4,
# 9 + 8, 10 + 9), three (8 + 8 + 4), four (8 + 8 + 8 + 1)
@pytest.mark.parametrize("tokens", [1025, 1088, 1089, 1152, 1153, 1280, 2600, 2817, 2880, 3009, 4120, 4700, 5000, 6300])
def test_rows_do_not_depend_on_the_tile(tokens):
    from rl_engine import _C

    vocab, hidden = 2060, 128
    gen = torch.Generator(device="cuda").manual_seed(tokens)
    h = torch.randn((tokens, hidden), generator=gen, device="cuda", dtype=torch.bfloat16)
    w = torch.randn((vocab, hidden), generator=gen, device="cuda", dtype=torch.bfloat16).mul_(0.2)
    ids = torch.randint(0, vocab - 60, (tokens,), generator=gen, device="cuda")
    extra = {
        "bias": torch.randn((vocab,), generator=gen, device="cuda"),
        "temperature": torch.empty(tokens, device="cuda").uniform_(0.6, 1.2, generator=gen),
    }
    logp, lse, logits = _C.fused_linear_logp(h, w, ids, return_logits=True, real_vocab_size=vocab - 60, **extra)
    plain = _C.fused_linear_logp(h, w, ids, real_vocab_size=vocab - 60, **extra)
    assert torch.equal(plain[0], logp) and torch.equal(plain[1], lse)
    for first in range(0, tokens, 777):
        part = slice(first, min(first + 777, tokens))
        few = dict(extra, temperature=extra["temperature"][part].contiguous())
        want = _C.fused_linear_logp(h[part].contiguous(), w, ids[part].contiguous(), return_logits=True, real_vocab_size=vocab - 60, **few)
        for got, exp in zip((logp, lse, logits), want):
            assert torch.equal(got[part].view(torch.int32), exp.view(torch.int32))
