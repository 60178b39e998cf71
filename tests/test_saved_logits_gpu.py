"""LogP backward from the logits the forward kept: the same bits as with the logits computed again."""

import pytest
import torch

from rl_engine import _C
from rl_engine.backends.rocm.logprob import linear_logp as module
from rl_engine.ops.logprob import deterministic_linear_logp

pytestmark = pytest.mark.gpu


def _inputs(tokens, vocab, hidden, seed=7):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    h = torch.randn((tokens, hidden), generator=gen, device="cuda", dtype=torch.bfloat16)
    w = torch.randn((vocab, hidden), generator=gen, device="cuda", dtype=torch.bfloat16) * 0.05
    ids = torch.randint(0, vocab, (tokens,), generator=gen, device="cuda")
    g = torch.randn((2, tokens), generator=gen, device="cuda")
    return h, w, ids, g


# token counts of the few-token, stream-group and tiled forwards; vocabularies that 8 and 64 do and do not divide, below
# and above one 4096-column chunk of the elementwise pass and at its edges
@pytest.mark.parametrize("tokens", [1, 65, 300, 1025])
@pytest.mark.parametrize("vocab, real", [(8, 8), (1000, 997), (4096, 4096), (4099, 4099), (12289, 12000)])
def test_same_bits(tokens, vocab, real):
    h, w, ids, g = _inputs(tokens, vocab, 128)
    ids = ids.clamp(max=real - 1)
    temperature = torch.linspace(0.6, 1.3, tokens, device="cuda")
    bias = torch.linspace(-1, 1, vocab, device="cuda")
    for bias_arg, temp_arg in ((None, None), (bias, temperature)):
        logits = torch.full((tokens, _C.linear_logp_logits_row_stride(vocab)), float("nan"), device="cuda")
        logp, lse = _C.fused_linear_logp_into(h, w, ids, bias_arg, temp_arg, real, logits)
        plain = _C.fused_linear_logp(h, w, ids, bias_arg, temp_arg, False, real)
        assert torch.equal(logp, plain[0]) and torch.equal(lse, plain[1])
        for need_bias in (False, True):
            want = _C.fused_linear_logp_bwd(h, w, ids, lse, g[0], g[1], bias_arg, temp_arg, real, need_grad_bias=need_bias)
            got = _C.fused_linear_logp_bwd(
                h, w, ids, lse, g[0], g[1], bias_arg, temp_arg, real, need_grad_bias=need_bias, logits=logits
            )
            for a, b in zip(got, want):
                assert (a is None) == (b is None) and (a is None or torch.equal(a, b))


def _saved_and_gradients(h, w, ids, g):
    h, w = h.clone().requires_grad_(), w.clone().requires_grad_()
    logp, _ = deterministic_linear_logp(h, w, ids)
    node = logp.grad_fn.next_functions[0][0]  # behind the reshape to the leading dimensions
    saved = [t for t in node.saved_tensors if t is not None and t.dim() == 2 and t.dtype == torch.float32]
    first = torch.autograd.grad(logp, (h, w), g[0], retain_graph=True)
    again = torch.autograd.grad(logp, (h, w), g[0])
    assert all(torch.equal(a, b) for a, b in zip(first, again))
    return len(saved), first


def test_what_is_saved(monkeypatch):
    """On the device, with its own answers about its memory."""
    h, w, ids, g = _inputs(module._SAVED_LOGITS_MIN_TOKENS, 1031, module._SAVED_LOGITS_MIN_HIDDEN)
    kept, grads = _saved_and_gradients(h, w, ids, g)
    assert kept == 1
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, lambda t: t):
        hooked, want = _saved_and_gradients(h, w, ids, g)
    assert hooked == 0 and all(torch.equal(a, b) for a, b in zip(grads, want))
    for name, value in (
        ("_SAVED_LOGITS_MAX_BYTES", 4 * h.size(0) * 1031),
        ("_SAVED_LOGITS_MIN_HIDDEN", h.size(1) + 1),
        ("_SAVED_LOGITS_MIN_TOKENS", h.size(0) + 1),
    ):
        with monkeypatch.context() as patch:
            patch.setattr(module, name, value)
            count, want = _saved_and_gradients(h, w, ids, g)
            assert count == 0 and all(torch.equal(a, b) for a, b in zip(grads, want))
    # switched off, and with little memory left (tests/test_saved_logits_memory.py has the limits themselves)
    with module.recompute_logits():
        count, want = _saved_and_gradients(h, w, ids, g)
    assert count == 0 and all(torch.equal(a, b) for a, b in zip(grads, want))
    monkeypatch.setattr(module, "_SAVED_LOGITS_UNCHECKED_BYTES", 0)
    monkeypatch.setattr(torch.cuda, "mem_get_info", lambda device: (1 << 20, 1 << 20))
    count, want = _saved_and_gradients(h, w, ids, g)
    assert count == 0 and all(torch.equal(a, b) for a, b in zip(grads, want))
