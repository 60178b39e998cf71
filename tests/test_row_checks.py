"""The value checks of the from-logits entry: what they refuse before anything reaches the device."""

from __future__ import annotations

from contextlib import nullcontext

import pytest
import torch

from rl_engine import _C


def test_refused_under_graph_capture(monkeypatch):
    """Their answer is read back, and a replay would write to host memory that is gone by then."""
    launched = []
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
    monkeypatch.setattr(_C, "_on", lambda device: nullcontext())
    monkeypatch.setattr(_C._lib, "load", lambda: launched.append("library"))
    with pytest.raises(RuntimeError, match="captured"):
        _C.RowChecks(torch.zeros(4, dtype=torch.long), 0, 8)
    assert not launched


@pytest.mark.gpu
def test_a_capture_goes_on_after_the_refusal():
    from rl_engine.ops.logprob import deterministic_logp_from_logits

    z = torch.randn(6, 640, device="cuda")
    ids = torch.arange(6, device="cuda")
    want = deterministic_logp_from_logits(z, ids)
    x = torch.ones(64, device="cuda")
    x + 1
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        with pytest.raises(RuntimeError, match="captured"):
            deterministic_logp_from_logits(z, ids)
        y = x + 1
    for start in (3.0, 5.0):
        x.fill_(start)
        graph.replay()
        torch.cuda.synchronize()
        assert bool((y == start + 1).all())
    assert all(torch.equal(a, b) for a, b in zip(want, deterministic_logp_from_logits(z, ids)))


@pytest.mark.gpu
def test_no_rows_have_nothing_to_check(monkeypatch):
    """No launch, no host memory and no wait; the temperature's size still counts."""
    from rl_engine.ops.logprob import deterministic_logp_from_logits

    def unused(*args):
        raise AssertionError("nothing to check")

    monkeypatch.setattr(_C, "RowChecks", unused)
    z, ids = torch.empty((0, 640), device="cuda"), torch.empty(0, dtype=torch.long, device="cuda")
    for temperature in (None, 0.7, torch.empty(0)):
        logp, lse = deterministic_logp_from_logits(z, ids, temperature=temperature)
        assert logp.shape == lse.shape == (0,)
    with pytest.raises(ValueError, match="temperature"):
        deterministic_logp_from_logits(z, ids, temperature=torch.ones(3))
