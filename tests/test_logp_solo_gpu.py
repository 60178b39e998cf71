"""Linear-LogP with one wave per SIMD: the bits of the small token tiles (log-probs, log-sum-exp, stored logits) at the edges of its
units - one to four vocabulary tiles of a split, a last token tile of 1 to 255 tokens beside and behind the whole ones, padded and
ragged vocabularies - and nothing written beside the logits."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda"


def _same(a, b):
    return torch.equal(a.contiguous().view(torch.int32), b.contiguous().view(torch.int32))


# (tokens, vocabulary, hidden, real vocabulary): units of 192 to 320 (whole round and more of 256 CUs), 1 ... 4 tiles in the last split
@pytest.mark.parametrize(
    "tokens,vocab,hidden,real",
    [(1024 + 1, 50000, 64, 50000), (1280 + 64, 45001, 64, 44900), (1536 + 65, 40704, 128, 40704), (2048 + 128, 32769, 64, 32769),
     (2048 + 129, 33024, 64, 32000), (2303, 28672, 192, 28672), (4096, 17000, 64, 16999), (4096 + 30, 16641, 64, 16641),
     (3072 + 100, 25000, 64, 25000), (3072 + 1, 25473, 128, 25400), (2048 + 64, 40001, 64, 40001)],
)  # fmt: skip
@pytest.mark.parametrize("temperature", [False, True])
def test_same_bits_as_the_small_token_tiles(tokens, vocab, hidden, real, temperature):
    from rl_engine import _C, _lib

    gen = torch.Generator(device=DEV).manual_seed(tokens + vocab)
    h = torch.randn((tokens, hidden), generator=gen, device=DEV, dtype=torch.bfloat16)
    w = torch.randn((vocab, hidden), generator=gen, device=DEV, dtype=torch.bfloat16).mul_(0.1)
    ids = torch.randint(0, real, (tokens,), generator=gen, device=DEV)
    ids[:3] = torch.tensor([0, real - 1, real // 2], device=DEV)
    t = torch.rand(tokens, generator=gen, device=DEV) + 0.5 if temperature else None
    small = _lib.LOGP_CONFIGS["128"]
    want = _C.fused_linear_logp(h, w, ids, None, t, True, real, config=small)
    got = _C.fused_linear_logp(h, w, ids, None, t, True, real)
    plain = _C.fused_linear_logp(h, w, ids, None, t, False, real)
    for a, b in zip(got, want):
        assert _same(a, b)
    assert _same(plain[0], want[0]) and _same(plain[1], want[1])


def test_targets_of_another_shard_and_strided_logits():
    from rl_engine import _C, _lib

    tokens, vocab, hidden, start = 2048 + 50, 33000, 64, 1000
    gen = torch.Generator(device=DEV).manual_seed(1)
    h = torch.randn((tokens, hidden), generator=gen, device=DEV, dtype=torch.bfloat16)
    w = torch.randn((vocab, hidden), generator=gen, device=DEV, dtype=torch.bfloat16).mul_(0.1)
    ids = torch.randint(0, vocab + 3000, (tokens,), generator=gen, device=DEV)
    out = [_C.fused_linear_logp(h, w, ids, None, None, False, vocab, vocab_start_index=start, config=c) for c in (0, _lib.LOGP_CONFIGS["128"])]
    for a, b in zip(*out):
        assert _same(a, b)
    outside = (ids < start) | (ids >= start + vocab)
    assert bool(torch.isnan(out[0][0][outside]).all()) and not bool(torch.isnan(out[0][0][~outside]).any())


@pytest.mark.parametrize("vocab", [33001, 33088, 40001, 40064])
def test_kept_logits_are_the_returned_ones_and_end_at_the_vocabulary(vocab):
    from rl_engine import _C

    tokens, hidden = 2048 + 50, 64
    gen = torch.Generator(device=DEV).manual_seed(vocab)
    h = torch.randn((tokens, hidden), generator=gen, device=DEV, dtype=torch.bfloat16)
    w = torch.randn((vocab, hidden), generator=gen, device=DEV, dtype=torch.bfloat16).mul_(0.1)
    ids = torch.randint(0, vocab, (tokens,), generator=gen, device=DEV)
    kept = torch.full((tokens, _C.linear_logp_logits_row_stride(vocab)), 7.0, device=DEV)
    logp, lse = _C.fused_linear_logp_into(h, w, ids, None, None, vocab, kept)
    # rows of an odd vocabulary are not 16-byte aligned: the eight-wave loop returns those
    want = _C.fused_linear_logp(h, w, ids, None, None, True, vocab)
    assert _same(logp, want[0]) and _same(lse, want[1]) and _same(kept[:, :vocab], want[2])
    assert bool((kept[:, vocab:] == 7.0).all())
