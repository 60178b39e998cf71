"""The fused gate/up projection of 17 to 128 tokens (csrc/swiglu.hip: det_gemm_swiglu_few_kernel): the projection followed by
the activation, bit for bit, for every tile width around its edges, and nothing written beside the result."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda"


# intermediate sizes for tiles of 16, 32, 48 and 64 features: whole, ragged by one and by less than a store
@pytest.mark.parametrize("inter", [16, 100, 4096, 4097, 8190, 8208, 12288, 12283, 12400])
@pytest.mark.parametrize("tokens", [16, 17, 63, 64, 65, 96, 97, 128, 129])
def test_projection_and_activation_in_one(tokens, inter):
    from rl_engine import _C

    gen = torch.Generator(device=DEV).manual_seed(tokens + inter)
    x = torch.randn((tokens, 512), generator=gen, device=DEV, dtype=torch.bfloat16)
    w = torch.randn((2 * inter, 512), generator=gen, device=DEV, dtype=torch.bfloat16).mul_(0.1)
    pad = torch.full((tokens + 1, inter + 5), 7.0, device=DEV, dtype=torch.bfloat16)
    _C.det_gemm_swiglu(x, w, pad[:tokens, :inter])
    gate_up = torch.empty((tokens, 2 * inter), device=DEV, dtype=torch.bfloat16)
    _C.gemm_strided(x, w.t(), gate_up)
    want = _C.swiglu_packed_forward(gate_up).view(torch.int16)
    assert torch.equal(pad[:tokens, :inter].contiguous().view(torch.int16), want)
    assert bool((pad[tokens] == 7.0).all()) and bool((pad[:, inter:] == 7.0).all())
    assert torch.equal(_C.det_gemm_swiglu(x, w).view(torch.int16), want)


# one intermediate size of each tile width (16, 32, 48 and 64 features), both tile heights; reductions below the rule, of fewer
# stages than the ring holds, of as many and of more (a slot is used again)
@pytest.mark.parametrize("tokens", [40, 100])
@pytest.mark.parametrize("inter", [3000, 4096, 8190, 12283, 12400])
@pytest.mark.parametrize("k", [64, 384, 448, 512, 640, 896, 1024, 1152, 2048, 4096])
def test_reduction_lengths_around_the_rule(k, inter, tokens):
    from rl_engine import _C

    gen = torch.Generator(device=DEV).manual_seed(k)
    x = torch.randn((tokens, k), generator=gen, device=DEV, dtype=torch.bfloat16)
    w = torch.randn((2 * inter, k), generator=gen, device=DEV, dtype=torch.bfloat16).mul_(0.05)
    gate_up = torch.empty((tokens, 2 * inter), device=DEV, dtype=torch.bfloat16)
    _C.gemm_strided(x, w.t(), gate_up)
    assert torch.equal(_C.det_gemm_swiglu(x, w).view(torch.int16), _C.swiglu_packed_forward(gate_up).view(torch.int16))
    # infinities and NaN stay in their rows
    x[3] = float("inf")
    x[7, 0] = float("nan")
    _C.gemm_strided(x, w.t(), gate_up)
    want, got = _C.swiglu_packed_forward(gate_up), _C.det_gemm_swiglu(x, w)
    nan = torch.isnan(want)
    assert torch.equal(torch.isnan(got), nan)
    assert torch.equal(torch.where(nan, 0, got.view(torch.int16)), torch.where(nan, 0, want.view(torch.int16)))
