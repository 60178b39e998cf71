"""The native host side answers None to what is not everyday (CPU tensors, wrong types, counts), so that the general way words
the errors, and is bound to the loaded library."""

from __future__ import annotations

import pytest
import torch


def test_cpu_tensors_and_other_objects_are_not_everyday(rlk_lib):
    from rl_engine import _host

    native = _host.native()
    x, w = torch.zeros(4, 8, dtype=torch.bfloat16), torch.zeros(8, 8, dtype=torch.bfloat16)
    assert native.linear(x, w) is None and native.linear(x, None) is None and native.linear(x) is None
    assert native.packed_ffn(x, w, w) is None and native.ffn(x, w, w, w) is None
    f = torch.zeros(2, 3)
    assert native.grpo(f, f, f, torch.zeros(2), None, 0.2, 0.0) is None
    assert native.grpo(f, f, f, torch.zeros(2), None, "0.2", 0.0) is None
    assert native.grpo(f, f, f, torch.zeros(2), None, 0.2, f) is None


def test_the_entry_points_still_word_their_errors():
    from rl_engine.ops.ffn import qwen3_ffn, qwen3_ffn_packed_inference
    from rl_engine.ops.gemm import DetGemmOp
    from rl_engine.ops.loss import grpo_ratio_kl_loss

    x = torch.zeros(4, 8, dtype=torch.bfloat16)
    with pytest.raises(AssertionError, match="Inputs must be on ROCm device"):
        DetGemmOp().linear(x, x)
    with pytest.raises(AssertionError, match="BF16 only"):
        DetGemmOp().linear(x.float(), x.float())
    with pytest.raises(TypeError, match="dtype bfloat16"):
        qwen3_ffn_packed_inference(x.float(), x, x)
    with pytest.raises(ValueError, match="must have shape"):
        qwen3_ffn(x, x, x, x)
    with pytest.raises(ValueError, match="one shape"):
        grpo_ratio_kl_loss(torch.zeros(2, 3), torch.zeros(2, 4), torch.zeros(2, 3), torch.zeros(2))


def test_bind_refuses_a_library_without_an_entry_point():
    from rl_engine import _torch_host

    with pytest.raises(RuntimeError, match="rlk_last_error"):
        _torch_host.bind({}, None, None, None)
