"""Gradients of a linear layer: the direct call for everyday operands and the general one give the same bits."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda"


def _form(t: torch.Tensor, form: str) -> torch.Tensor:
    rows, cols = t.shape
    if form == "plain":
        return t
    if form == "pitch":  # rows inside a wider buffer, still 16-byte aligned
        wide = torch.zeros((rows, cols + 24), dtype=t.dtype, device=t.device)
        wide[:, :cols] = t
        return wide[:, :cols]
    if form == "odd_pitch":
        wide = torch.zeros((rows, cols + 3), dtype=t.dtype, device=t.device)
        wide[:, :cols] = t
        return wide[:, :cols]
    if form == "offset":  # rows that start 2 bytes past an aligned address
        flat = torch.zeros((rows * cols + 1,), dtype=t.dtype, device=t.device)
        flat[1:] = t.reshape(-1)
        return flat[1:].view(rows, cols)
    if form == "transposed":
        return t.t().contiguous().t()
    assert form == "one_row_repeated"
    return t[:1].expand(rows, cols)


@pytest.mark.parametrize("form", ["plain", "pitch", "odd_pitch", "offset", "transposed", "one_row_repeated"])
@pytest.mark.parametrize("operand", ["grad", "other"])
@pytest.mark.parametrize("tokens,inputs,outputs", [(1, 64, 128), (67, 136, 200), (130, 100, 72), (70, 1, 8)])
def test_same_bits_as_the_general_call(form, operand, tokens, inputs, outputs):
    from rl_engine import _C
    from rl_engine.backends.rocm.gemm import det_gemm

    gen = torch.Generator(device=DEV).manual_seed(tokens + inputs)
    rand = lambda *shape: torch.randn(shape, generator=gen, device=DEV, dtype=torch.bfloat16)  # noqa: E731
    x, w, g = rand(tokens, inputs), rand(outputs, inputs), rand(tokens, outputs)
    if operand == "grad":
        g = _form(g, form)
    else:
        x, w = _form(x, form), _form(w, form)
    dx = det_gemm.mfma_linear_input_gradient(g, w)
    dw = det_gemm.mfma_linear_weight_gradient(x, g)
    want_dx, want_dw = torch.empty_like(dx), torch.empty_like(dw)
    # whole copies with the reduction contiguous: the general kernel path
    _C.gemm_strided(g.contiguous(), w.t().contiguous().t(), want_dx)
    _C.gemm_strided(g.t().contiguous(), x.t().contiguous().t(), want_dw)
    assert dx.shape == (tokens, inputs) and dw.shape == (outputs, inputs)
    assert torch.equal(dx.view(torch.int16), want_dx.view(torch.int16))
    assert torch.equal(dw.view(torch.int16), want_dw.view(torch.int16))


def test_what_was_refused_stays_refused():
    from rl_engine.backends.rocm.gemm import det_gemm

    g = torch.zeros((4, 16), device=DEV, dtype=torch.bfloat16)
    w = torch.zeros((16, 8), device=DEV, dtype=torch.bfloat16)
    with pytest.raises(ValueError, match="K mismatch"):
        det_gemm.mfma_linear_input_gradient(g, w[:8])
    with pytest.raises(TypeError, match="BF16"):
        det_gemm.mfma_linear_input_gradient(g, w.float())
    with pytest.raises(ValueError, match="K mismatch"):
        det_gemm.mfma_linear_weight_gradient(w[:2].contiguous(), g)
    with pytest.raises(RuntimeError, match="share one ROCm device"):
        det_gemm.mfma_linear_input_gradient(g, w.cpu())
