"""The GRPO kernels at the sizes where their loops turn: forward sums and the one-pass backward on a real MI355X."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda"


def _case(rollouts, tokens, seed, with_mask):
    g = torch.Generator().manual_seed(seed)
    cur = -torch.randn((rollouts, tokens), generator=g).abs()
    old = cur + 0.3 * torch.randn((rollouts, tokens), generator=g)
    ref = cur + 0.2 * torch.randn((rollouts, tokens), generator=g)
    adv = torch.randn(rollouts, generator=g)
    mask = torch.rand((rollouts, tokens), generator=g) < 0.7 if with_mask else None
    return cur, old, ref, adv, mask


# one thread's token, the 256-token stride, four strides in flight, the backward's 1024-token chunk; the finish
# kernel's 256 sequences at a time
@pytest.mark.parametrize("rollouts,tokens", [(1, 1), (2, 255), (3, 257), (5, 1023), (2, 1025), (1, 2049), (255, 3), (257, 5), (600, 1)])
@pytest.mark.parametrize("with_mask", [False, True])
def test_forward_sums_and_backward_at_loop_edges(rollouts, tokens, with_mask):
    from rl_engine.ops.loss import grpo_ratio_kl_loss

    cur, old, ref, adv, mask = _case(rollouts, tokens, 31 * rollouts + tokens, with_mask)
    on_gpu = [t.to(DEV) if t is not None else None for t in (old, ref, adv, mask)]
    x = cur.to(DEV).requires_grad_(True)
    out = grpo_ratio_kl_loss(x, *on_gpu, clip_eps=0.2, beta=0.3)
    weights = (0.7, -0.4, 1.3)
    total = weights[0] * out.loss + weights[1] * out.policy_loss + weights[2] * out.kl
    (grad,) = torch.autograd.grad(total, x)

    z = cur.double().requires_grad_(True)
    keep = torch.ones_like(z) if mask is None else mask.double()
    count = keep.sum().clamp(min=1e-8)
    ratio, d = torch.exp(z - old.double()), ref.double() - z
    a = adv.double()[:, None]
    terms = -torch.minimum(ratio * a, ratio.clamp(0.8, 1.2) * a) * keep
    policy, kl = terms.sum() / count, ((torch.exp(d) - d - 1) * keep).sum() / count
    loss = policy + 0.3 * kl
    (want,) = torch.autograd.grad(weights[0] * loss + weights[1] * policy + weights[2] * kl, z)

    # fp32 sums of n terms: n 2^-24 of the sum of magnitudes bounds any order; a term carries a few roundings more
    # (exp of a difference of magnitude up to 8, with its own rounding: 2^-20)
    n = rollouts * tokens
    bound = (n * 2.0**-24 + 2.0**-20) * float(terms.detach().abs().sum() / count) + 1e-12
    assert abs(float(out.policy_loss.detach()) - float(policy.detach())) <= bound
    kl_bound = (n * 2.0**-24 + 2.0**-20) * float(((torch.exp(d) + d.abs() + 1) * keep).detach().sum() / count) + 1e-12
    assert abs(float(out.kl.detach()) - float(kl.detach())) <= kl_bound
    per_token = float(a.abs().max()) * float(ratio.detach().max()) + 2 + float(torch.exp(d.detach()).max())
    assert (grad.cpu().double() - want).abs().max().item() <= 2.0**-19 * 3 * per_token / float(count)
    if mask is not None:
        assert bool((grad.cpu()[~mask] == 0).all())


def test_backward_kernel_equals_the_differentiable_form():
    """create_graph=True runs the elementwise form (and can be differentiated again): the kernel's values, bit for bit."""
    from rl_engine.ops.loss import grpo_ratio_kl_loss

    cur, old, ref, adv, mask = (t.to(DEV) for t in _case(7, 1300, 77, True))
    grads = []
    for create_graph in (False, True):
        x = cur.clone().requires_grad_(True)
        out = grpo_ratio_kl_loss(x, old, ref, adv, mask, clip_eps=0.15, beta=0.05)
        (grad,) = torch.autograd.grad(out.loss, x, create_graph=create_graph)
        grads.append(grad)
    assert torch.equal(grads[0].view(torch.int32), grads[1].detach().view(torch.int32))
    (second,) = torch.autograd.grad(grads[1].sum(), x)
    assert bool(torch.isfinite(second).all()) and float(second.abs().max()) > 0


@pytest.mark.parametrize("layout", ["column_slice", "transposed"])
def test_strided_log_probs_can_be_differentiated_twice(layout):
    """Log-probs that are not contiguous (a slice without the last token, a transpose): both orders of gradient are
    those of the contiguous copy, bit for bit."""
    from rl_engine.ops.loss import grpo_ratio_kl_loss

    cur, old, ref, adv, mask = (t.to(DEV) for t in _case(5, 301, 78, True))
    results = []
    for strided in (False, True):
        x = cur.clone()
        if strided and layout == "column_slice":
            x = torch.cat([x, x[:, :1]], dim=1)[:, :-1]
        elif strided:
            x = x.t().contiguous().t()
        assert x.is_contiguous() != strided
        x = x.detach().requires_grad_(True)
        out = grpo_ratio_kl_loss(x, old, ref, adv, mask, clip_eps=0.2, beta=0.1)
        (plain,) = torch.autograd.grad(out.loss, x, retain_graph=True)
        (grad,) = torch.autograd.grad(out.loss, x, create_graph=True)
        (second,) = torch.autograd.grad(grad.square().sum(), x)
        results.append([t.detach().contiguous().view(torch.int32) for t in (plain, grad, second)])
    for a, b in zip(*results):
        assert torch.equal(a, b)
