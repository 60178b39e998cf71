"""LogP from logits on a real MI355X: the streamed gradient stores of large calls and the device-side value checks."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda"


# 128 MiB of gradient is where the stores change: just above it, in rows that are whole 16-byte vectors and in rows
# that are not (every row then has another alignment and an element-wise end)
@pytest.mark.parametrize("dtype,rows,vocab", [
    (torch.bfloat16, 445, 151936), (torch.bfloat16, 1040, 65531), (torch.float16, 1030, 65536), (torch.float32, 1025, 32773),
])  # fmt: skip
def test_streamed_gradient_equals_the_same_rows_alone(dtype, rows, vocab):
    from rl_engine import _C

    gen = torch.Generator(device=DEV).manual_seed(rows)
    z = torch.randn((rows, vocab), generator=gen, device=DEV).to(dtype)
    assert z.numel() * z.element_size() >= 128 << 20
    target = torch.randint(0, vocab, (rows,), generator=gen, device=DEV)
    lse = torch.logsumexp(z[:, :1000].float(), dim=1)
    g_logp, g_lse = (torch.randn(rows, generator=gen, device=DEV) for _ in range(2))
    whole = _C.hip_deterministic_logp_backward(z, lse, g_logp, g_lse, target, 0, vocab - 3, True)
    for lo, hi in ((0, 3), (rows // 2, rows // 2 + 2), (rows - 3, rows)):
        part = [t[lo:hi].contiguous() for t in (lse, g_logp, g_lse, target)]
        alone = _C.hip_deterministic_logp_backward(z[lo:hi], part[0], part[1], part[2], part[3], 0, vocab - 3, True)
        bits = torch.int32 if dtype == torch.float32 else torch.int16
        assert torch.equal(whole[lo:hi].view(bits), alone.view(bits))
    assert not bool(whole[:, vocab - 3 :].any())  # padded columns


@pytest.mark.parametrize("rows", [1, 63, 256, 257, 64 * 256 + 1])
def test_row_checks_find_the_one_bad_value(rows):
    from rl_engine import _C

    good = torch.randint(5, 90, (rows,), device=DEV)
    warm = torch.full((rows,), 0.5, device=DEV)
    assert _C.RowChecks(good, 5, 90).results() == (False, False)
    assert _C.RowChecks(good, 5, 90, warm).results() == (False, False)
    for at in {0, rows // 2, rows - 1}:
        for value in (4, 90, -1):
            bad = good.clone()
            bad[at] = value
            assert _C.RowChecks(bad, 5, 90, warm).results() == (True, False)
        cold = warm.clone()
        cold[at] = 0.0
        assert _C.RowChecks(good, 5, 90, cold).results() == (False, True)


def test_a_rejected_call_leaves_nothing_behind():
    """The forward runs behind the checks, so it also ran for the call that raises: the next call is not affected."""
    from rl_engine.ops.logprob import deterministic_logp_from_logits

    z = torch.randn(6, 640, device=DEV)
    ids = torch.arange(6, device=DEV)
    want = deterministic_logp_from_logits(z, ids)
    for wrong, temperature in ((640, None), (-1, None), (3, 0.0)):
        bad = ids.clone()
        bad[2] = wrong
        with pytest.raises(ValueError):
            deterministic_logp_from_logits(z, bad, temperature=temperature)
        again = deterministic_logp_from_logits(z, ids)
        assert all(torch.equal(a, b) for a, b in zip(want, again))


# logits of more than 232 MiB: their first workgroups read past the caches, the split lying inside a row, at a row and
# (several column groups) inside a group
@pytest.mark.parametrize("dtype,rows,vocab", [
    (torch.bfloat16, 812, 151936), (torch.bfloat16, 1700, 151936), (torch.float16, 20000, 6400), (torch.float32, 950, 65536),
])  # fmt: skip
@pytest.mark.parametrize("temperature", [None, 0.7])
def test_streamed_forward_equals_the_same_rows_alone(dtype, rows, vocab, temperature):
    from rl_engine.ops.logprob import deterministic_logp_from_logits

    gen = torch.Generator(device=DEV).manual_seed(rows)
    z = torch.randn((rows, vocab), generator=gen, device=DEV).to(dtype)
    assert z.numel() * z.element_size() > 232 << 20
    ids = torch.randint(0, vocab, (rows,), generator=gen, device=DEV)
    whole = deterministic_logp_from_logits(z, ids, temperature=temperature)
    for lo in range(0, rows, 256):
        part = deterministic_logp_from_logits(z[lo : lo + 256], ids[lo : lo + 256], temperature=temperature)
        for a, b in zip(whole, part):
            assert torch.equal(a[lo : lo + 256].view(torch.int32), b.view(torch.int32))
