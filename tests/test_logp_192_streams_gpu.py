"""Fused linear-LogP on 192-token stream groups: the bits of the other tiles around their edges, with and without logits,
and at the sizes whose automatic choice they are."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tokens", [1, 191, 192, 193, 385, 577])
@pytest.mark.parametrize("vocab", [500, 2048, 2060])
def test_same_bits_as_the_64_token_tiles(tokens, vocab):
    from rl_engine import _C, _lib

    gen = torch.Generator(device="cuda").manual_seed(tokens + vocab)
    h = torch.randn((tokens, 192), generator=gen, device="cuda", dtype=torch.bfloat16)
    w = torch.randn((vocab, 192), generator=gen, device="cuda", dtype=torch.bfloat16).mul_(0.1)
    ids = torch.randint(0, vocab, (tokens,), generator=gen, device="cuda")
    bias = torch.randn((vocab,), generator=gen, device="cuda")
    temperature = torch.empty(tokens, device="cuda").uniform_(0.6, 1.2, generator=gen)
    for extra in ({}, {"bias": bias, "temperature": temperature, "real_vocab_size": vocab - 3}):
        ids_ok = ids % (vocab - 3)
        got = _C.fused_linear_logp(h, w, ids_ok, config=_lib.LOGP_CONFIGS["192_streams"], **extra)
        want = _C.fused_linear_logp(h, w, ids_ok, config=_lib.LOGP_CONFIGS["64_streams"], **extra)
        auto = _C.fused_linear_logp(h, w, ids_ok, **extra)
        for a, b, c in zip(got, want, auto):
            if a is not None:
                assert torch.equal(a.view(torch.int32), b.view(torch.int32)) and torch.equal(c.view(torch.int32), b.view(torch.int32))


def test_stored_logits_of_192_token_tiles():
    from rl_engine import _C

    gen = torch.Generator(device="cuda").manual_seed(9)
    h = torch.randn((300, 128), generator=gen, device="cuda", dtype=torch.bfloat16)
    w = torch.randn((32768, 128), generator=gen, device="cuda", dtype=torch.bfloat16).mul_(0.1)
    ids = torch.randint(0, 32768, (300,), generator=gen, device="cuda")
    logits = _C.fused_linear_logp(h, w, ids, return_logits=True)[2]  # 300 tokens of this vocabulary are the 192-token tiles' choice
    want = torch.empty((300, 32768), device="cuda")
    _C.gemm_strided(h, w.t(), want)
    assert torch.equal(logits, want)
