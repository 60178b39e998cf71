"""What memory the kept logits of a differentiable linear-LogP may take: on CPU tensors, with the device's answers
replaced."""

from __future__ import annotations

import gc

import pytest
import torch

from rl_engine import _C
from rl_engine.backends.rocm.logprob import linear_logp as module

TOKENS, VOCAB = 256, 1031
ROW_BYTES = 4 * _C.linear_logp_logits_row_stride(VOCAB)
SIZE = TOKENS * ROW_BYTES
PLENTY = 1 << 40


@pytest.fixture
def device(monkeypatch):
    """A device with the given number of free bytes (and what the allocator holds beside it)."""

    def has(free, reserved=0, allocated=0, fraction=1.0):
        monkeypatch.setattr(torch.cuda, "mem_get_info", lambda device: (free, PLENTY))
        monkeypatch.setattr(torch.cuda, "memory_reserved", lambda device: reserved)
        monkeypatch.setattr(torch.cuda, "memory_allocated", lambda device: allocated)
        monkeypatch.setattr(torch.cuda, "get_per_process_memory_fraction", lambda device: fraction)

    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    monkeypatch.setattr(module, "_SAVED_LOGITS_UNCHECKED_BYTES", 0)
    has(PLENTY)
    gc.collect()
    return has


def _hidden():
    return torch.empty((TOKENS, module._SAVED_LOGITS_MIN_HIDDEN), dtype=torch.bfloat16)


def test_all_graphs_alive_share_one_limit(device, monkeypatch):
    """Several forwards before one backward: together they hold no more than the limit, and a freed one makes room."""
    monkeypatch.setattr(module, "_SAVED_LOGITS_MAX_BYTES", 3 * SIZE + SIZE // 2)
    held = [module._logits_to_save(_hidden(), VOCAB) for _ in range(5)]
    assert [t is not None for t in held] == [True, True, True, False, False]
    assert sum(4 * t.numel() for t in held if t is not None) <= module._SAVED_LOGITS_MAX_BYTES
    half = VOCAB // 2 + 5  # rows of whole 64 values: a little more than half a buffer
    assert 4 * TOKENS * _C.linear_logp_logits_row_stride(half) > SIZE // 2
    assert module._logits_to_save(_hidden(), half) is None
    assert module._logits_to_save(_hidden(), half - 64) is not None
    del held[0]
    gc.collect()
    again = module._logits_to_save(_hidden(), VOCAB)
    assert again is not None and module._logits_to_save(_hidden(), VOCAB) is None


def test_a_graph_gives_its_share_back(device, monkeypatch):
    """The share is held from the forward to the end of the graph: through a backward that keeps it, not past one that
    frees it, and not past a graph that is dropped."""
    monkeypatch.setattr(module, "_SAVED_LOGITS_MAX_BYTES", SIZE)

    class Keeps(torch.autograd.Function):
        @staticmethod
        def forward(ctx, x):
            ctx.save_for_backward(x, module._logits_to_save(_hidden(), VOCAB))
            return x * 1

        @staticmethod
        def backward(ctx, grad):
            return grad if ctx.saved_tensors[1] is not None else grad * 0

    x = torch.ones(2, requires_grad=True)

    def free():
        return module._logits_to_save(_hidden(), VOCAB) is not None

    y = Keeps.apply(x)
    assert not free()
    torch.autograd.grad(y.sum(), x, retain_graph=True)
    assert not free()
    (grad,) = torch.autograd.grad(y.sum(), x)
    assert bool((grad == 1).all()) and free()
    y = Keeps.apply(x)
    assert not free()
    del y
    gc.collect()
    assert free()


def test_only_what_the_driver_has_free_counts(device, monkeypatch):
    """The buffer and the bf16 d(logits) of its backward within a quarter of the free memory. What the allocator has
    cached may be pieces: asked for more than it has in one, it would give its whole cache back first."""
    enough = 4 * (SIZE + SIZE // 2)
    device(enough)
    assert module._logits_to_save(_hidden(), VOCAB) is not None
    asked = []
    monkeypatch.setattr(torch, "empty", lambda *a, **k: asked.append(a))
    hidden = torch.zeros((TOKENS, module._SAVED_LOGITS_MIN_HIDDEN), dtype=torch.bfloat16)
    device(enough - 1)
    assert module._logits_to_save(hidden, VOCAB) is None
    device(SIZE, reserved=PLENTY, allocated=0)
    assert module._logits_to_save(hidden, VOCAB) is None
    # a process that may use a share of the card only
    device(PLENTY, reserved=PLENTY // 2, fraction=0.5)
    assert module._logits_to_save(hidden, VOCAB) is None
    assert not asked


def test_an_allocation_that_fails_is_no_error(device, monkeypatch):
    monkeypatch.setattr(module, "_SAVED_LOGITS_MAX_BYTES", SIZE)
    hidden = _hidden()
    tried = []

    def fails(*args, **kwargs):
        tried.append(args)
        raise torch.cuda.OutOfMemoryError("out of memory")

    with monkeypatch.context() as patch:
        patch.setattr(torch, "empty", fails)
        assert module._logits_to_save(hidden, VOCAB) is None
    assert len(tried) == 1
    assert module._logits_to_save(hidden, VOCAB) is not None  # it did not count


def test_switched_off_for_a_block(device):
    with module.recompute_logits():
        assert module._logits_to_save(_hidden(), VOCAB) is None
    with pytest.raises(KeyError), module.recompute_logits():
        raise KeyError
    assert module._logits_to_save(_hidden(), VOCAB) is not None


@pytest.mark.parametrize("wrong", ["rows", "columns", "stride", "dtype", "device"])
def test_the_forward_refuses_a_buffer_that_it_would_write_past(wrong):
    """Refused by its shape, before anything reaches a device (the operands here are on none)."""
    hidden, weight = _hidden(), torch.empty((VOCAB, module._SAVED_LOGITS_MIN_HIDDEN), dtype=torch.bfloat16)
    columns = _C.linear_logp_logits_row_stride(VOCAB)
    logits = {
        "rows": torch.empty((TOKENS - 1, columns)),
        "columns": torch.empty((TOKENS, VOCAB)),
        "stride": torch.empty((columns, TOKENS)).t(),
        "dtype": torch.empty((TOKENS, columns), dtype=torch.bfloat16),
        "device": torch.empty((TOKENS, columns), device="meta"),
    }[wrong]
    with pytest.raises(RuntimeError, match="logits must be"):
        _C.fused_linear_logp_into(hidden, weight, torch.zeros(TOKENS, dtype=torch.long), None, None, VOCAB, logits)
