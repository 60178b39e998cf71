"""The streaming kernel's consumers read a stage's fragments under the products of the stage before: the bits of the one-wave
tile for one stage, for an even and an odd number of them, for a last stage that is not full, and for fewer than the ring
holds, whatever the number of consumers."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda"


@pytest.mark.parametrize("config,tokens", [("stream16", 1), ("stream16", 16), ("stream16_deep", 7), ("stream64", 17), ("stream64", 48), ("stream64", 64)])  # fmt: skip
@pytest.mark.parametrize("tiles", [1, 2, 3, 4, 5, 7, 8, 14, 15, 16, 17, 18, 19, 33])
def test_number_of_stages(config, tokens, tiles):
    from rl_engine import _C, _lib

    gen = torch.Generator(device=DEV).manual_seed(100 * tokens + tiles)
    x = torch.randn((tokens, 64 * tiles), generator=gen, device=DEV, dtype=torch.bfloat16)
    w = torch.randn((41, 64 * tiles), generator=gen, device=DEV, dtype=torch.bfloat16)
    for dtype, bits in ((torch.bfloat16, torch.int16), (torch.float32, torch.int32)):
        pad = torch.full((tokens + 1, 48), 7.0, dtype=dtype, device=DEV)
        want = torch.empty((tokens, 41), dtype=dtype, device=DEV)
        _C.gemm_strided(x, w.t(), pad[:tokens, :41], config=_lib.GEMM_CONFIGS[config])
        _C.gemm_strided(x, w.t(), want, config=_lib.GEMM_CONFIGS["16x16"])
        assert torch.equal(pad[:tokens, :41].contiguous().view(bits), want.view(bits))
        assert bool((pad[tokens] == 7.0).all()) and bool((pad[:, 41:] == 7.0).all())


@pytest.mark.parametrize("k", [1024, 1088, 1152, 1216])
def test_gated_panels(k):
    from rl_engine import _C, _lib

    gen = torch.Generator(device=DEV).manual_seed(k)
    x = torch.randn((16, k), generator=gen, device=DEV, dtype=torch.bfloat16)
    w = torch.randn((2 * 75, k), generator=gen, device=DEV, dtype=torch.bfloat16).mul_(0.1)
    # non-finite values stay in their rows: the zeros that go before the first stage meet no operand
    x[3, 5], x[9, k - 1] = float("inf"), float("nan")
    gate_up = torch.empty((16, 150), device=DEV, dtype=torch.bfloat16)
    _C.gemm_strided(x, w.t(), gate_up, config=_lib.GEMM_CONFIGS["16x16"])
    want, got = _C.swiglu_packed_forward(gate_up), _C.det_gemm_swiglu(x, w)
    nan = torch.isnan(want)
    assert torch.equal(torch.isnan(got), nan)
    assert torch.equal(torch.where(nan, 0, got.view(torch.int16)), torch.where(nan, 0, want.view(torch.int16)))
