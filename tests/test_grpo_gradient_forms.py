"""Which gradients of the GRPO loss the backward kernel serves: whatever is more than plain memory takes the tensor
operations, which hold for it. The kernels are stood in for by the same formula on the CPU."""

from __future__ import annotations

import pytest
import torch
import torch.autograd.forward_ad as fwd

from rl_engine.backends.rocm.loss import grpo

CLIP, BETA = 0.2, 0.1


def _scalars(cur, old, ref, adv, mask):
    keep = torch.ones_like(cur) if mask is None else mask.to(cur.dtype)
    ratio, d = torch.exp(cur - old), ref - cur
    k3 = torch.exp(d) - d - 1
    a = adv.reshape(-1, 1)
    terms = -torch.minimum(ratio * a, ratio.clamp(1 - CLIP, 1 + CLIP) * a)
    count = keep.sum().clamp(min=1e-8)
    policy, kl = (terms * keep).sum() / count, (k3 * keep).sum() / count
    return torch.stack([policy + BETA * kl, policy, kl]), ratio * keep, k3 * keep


@pytest.fixture
def kernel_calls(monkeypatch):
    """The two kernels on CPU tensors; returns the list of gradients that the backward kernel was asked for."""
    calls = []

    def forward(cur, old, ref, adv, mask, clip_eps, beta):
        with torch.no_grad():
            out3, ratio, k3 = _scalars(cur, old, ref, adv, mask)
        inputs = tuple(t.contiguous() for t in (cur, old, ref, adv))
        keep = mask.contiguous().view(torch.uint8) if mask is not None else None
        counts = (mask if mask is not None else torch.ones_like(cur)).sum(1, dtype=torch.float32)
        return [out3, ratio, k3, (*inputs, keep), torch.cat([torch.zeros(2 * cur.size(0)), counts])]

    def backward(inputs, workspace, g_loss, g_policy, g_kl, clip_eps, beta):
        calls.append((g_loss, g_policy, g_kl))
        shape = inputs[0].shape
        memory = []
        for t, dtype in zip((*inputs, g_loss, g_policy, g_kl), [torch.float32] * 4 + [torch.uint8] + [torch.float32] * 3):
            if t is not None:  # the kernel reads rows of values, whatever the tensor's own type and strides say
                assert t.dtype is dtype, "the kernel would read past the tensor"
                t = torch.from_numpy(t.detach().numpy())
                t = t.as_strided(shape, (shape[1], 1)) if t.dim() == 2 else t
            memory.append(t)
        grad = grpo._elementwise_gradient(*memory, clip_eps, beta)
        active = inputs[4].sum() if inputs[4] is not None else torch.tensor(shape.numel())
        return grad * active / workspace[2 * shape[0] :].sum()

    monkeypatch.setattr(grpo._C, "grpo_ratio_kl_loss_saved", forward)
    monkeypatch.setattr(grpo._C, "grpo_ratio_kl_loss_bwd", backward)
    return calls


def _case(seed=3, rollouts=3, tokens=17):
    g = torch.Generator().manual_seed(seed)
    cur = -torch.rand((rollouts, tokens), generator=g, dtype=torch.float32)
    old = cur + 0.3 * torch.randn(cur.shape, generator=g)
    ref = cur + 0.2 * torch.randn(cur.shape, generator=g)
    return cur, old, ref, torch.randn(rollouts, generator=g), torch.rand(cur.shape, generator=g) < 0.7


def _loss(x, rest):
    return grpo.grpo_ratio_kl_loss(x, *rest, clip_eps=CLIP, beta=BETA)


def test_a_plain_gradient_is_the_kernels(kernel_calls):
    cur, *rest = _case()
    x = cur.clone().requires_grad_(True)
    torch.autograd.grad(_loss(x, rest).loss, x)
    assert len(kernel_calls) == 1


def test_batched_gradients(kernel_calls):
    cur, *rest = _case()
    x = cur.clone().requires_grad_(True)
    out = _loss(x, rest)
    weights = torch.tensor([1.0, -2.5, 0.0, 7.0])
    for scalar in (out.loss, out.policy_loss, out.kl):
        (one,) = torch.autograd.grad(scalar, x, retain_graph=True)
        (many,) = torch.autograd.grad(scalar, x, weights, retain_graph=True, is_grads_batched=True)
        # one product by the weight more or less: 2 roundings of the value
        torch.testing.assert_close(many, weights[:, None, None] * one, rtol=2.0**-22, atol=1e-9)
    rows = torch.autograd.functional.jacobian(lambda t: torch.stack(_loss(t, rest)[:3]), cur, vectorize=True)
    plain = torch.autograd.functional.jacobian(lambda t: torch.stack(_loss(t, rest)[:3]), cur)
    torch.testing.assert_close(rows, plain, rtol=2.0**-22, atol=1e-9)


def test_the_tangent_of_an_incoming_gradient(kernel_calls):
    """The gradient is linear in the incoming one, so its tangent is the gradient for the incoming tangent."""
    cur, *rest = _case()
    x = cur.clone().requires_grad_(True)
    loss = _loss(x, rest).loss
    (want,) = torch.autograd.grad(loss, x, torch.tensor(3.0), retain_graph=True)
    with fwd.dual_level():
        (grad,) = torch.autograd.grad(loss, x, fwd.make_dual(torch.tensor(0.5), torch.tensor(3.0)))
        tangent = fwd.unpack_dual(grad).tangent
    assert tangent is not None
    torch.testing.assert_close(tangent, want, rtol=2.0**-22, atol=1e-9)


class _Tagged(torch.Tensor):
    pass


def _hooks(pack, unpack):
    return torch.autograd.graph.saved_tensors_hooks(pack, unpack)


def test_saved_tensors_that_hooks_hand_back(kernel_calls):
    """Hooks that keep the values but not the layout or the type, and hooks that round them."""
    cur, *rest = _case(rollouts=3, tokens=301)
    x = cur.clone().requires_grad_(True)
    (want,) = torch.autograd.grad(_loss(x, rest).loss, x)

    def gradient(pack, unpack):
        with _hooks(pack, unpack):
            loss = _loss(x, rest).loss
        return torch.autograd.grad(loss, x)[0]

    def turned(t):
        return t.t().contiguous().t() if t.dim() == 2 else t

    torch.testing.assert_close(gradient(lambda t: t, turned), want, rtol=2.0**-22, atol=1e-9)
    torch.testing.assert_close(gradient(lambda t: t, torch.Tensor.double), want, rtol=2.0**-19, atol=1e-9)
    torch.testing.assert_close(gradient(lambda t: t, lambda t: t.as_subclass(_Tagged)), want, rtol=2.0**-22, atol=1e-9)
    assert len(kernel_calls) == 1  # the gradient to compare with

    # values rounded to bf16: the gradient of the rounded values, over the tokens that are really there
    def rounded(t):
        return t.to(torch.bfloat16).to(t.dtype) if t.is_floating_point() else t

    y = rounded(cur).requires_grad_(True)
    near = [rounded(t) for t in rest[:3]] + rest[3:]
    (want,) = torch.autograd.grad(_loss(y, near).loss, y)
    torch.testing.assert_close(gradient(rounded, lambda t: t), want, rtol=2.0**-22, atol=1e-9)


def test_mask_bytes_other_than_one_weigh_one(kernel_calls):
    """A bool tensor made from bytes may hold any of them: the differentiable form weighs a kept token with one, as the
    kernels do."""
    cur, old, ref, adv, mask = _case()
    want = grpo._elementwise_gradient(cur, old, ref, adv, mask.view(torch.uint8), torch.tensor(1.0), None, None, CLIP, BETA)
    got = grpo._elementwise_gradient(cur, old, ref, adv, mask.to(torch.uint8) * 255, torch.tensor(1.0), None, None, CLIP, BETA)
    assert torch.equal(got, want)
