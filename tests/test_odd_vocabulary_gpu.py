"""Gradients over vocabularies that no 16-byte chunk divides: the bits of the element-wise loops."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda"


# vocabularies that end one before, one behind and in the middle of a chunk, a store run and a row of d(logits); tokens of
# the few-token weight gradient (64, 128), one that no tile divides, and of the transposed hidden states (from 512)
@pytest.mark.parametrize("vocab", [1001, 1023, 1025, 2047, 2055, 3083])
@pytest.mark.parametrize("tokens", [1, 40, 64, 128, 200, 515])
def test_odd_vocabulary_backward(vocab, tokens):
    from rl_engine import _C, _lib

    gen = torch.Generator(device=DEV).manual_seed(vocab + tokens)
    h = torch.randn((tokens, 256), generator=gen, device=DEV).to(torch.bfloat16)
    w = (0.2 * torch.randn((vocab, 256), generator=gen, device=DEV)).to(torch.bfloat16)
    target = torch.randint(0, vocab, (tokens,), generator=gen, device=DEV)
    grad = torch.randn((tokens,), generator=gen, device=DEV)
    _, lse = _C.fused_linear_logp(h, w, target, None, None, False, vocab)
    got = []
    for config in (0, _lib.FORCE_STAGED):
        # what a workspace that is allocated next finds behind the vocabulary must not matter
        stale = torch.full((tokens * (vocab + 64),), float("nan"), dtype=torch.bfloat16, device=DEV)
        del stale
        got.append(_C.fused_linear_logp_bwd(h, w, target, lse, grad, grad, None, None, vocab, need_grad_bias=False, config=config))
    for fast, plain in zip(*got):
        if plain is not None:
            assert bool(torch.isfinite(fast).all())
            assert torch.equal(fast.view(torch.int16), plain.view(torch.int16))
