"""The 192-token tiles (256 x 192 and 192 x 192) at their edges: the bits of the other tiles for every operand layout that
reaches them, in the fused gate/up as well, and nothing written beside the result."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda"
# (tokens, outputs, K): one token, a tile, one more, whole and ragged tiles of both axes, the shortest reductions
SHAPES = [(1, 16, 64), (191, 255, 64), (192, 256, 128), (193, 257, 192), (385, 512, 256), (577, 200, 4096), (200, 777, 64)]


def _operands(shape, seed):
    m, n, k = shape
    gen = torch.Generator(device=DEV).manual_seed(seed)
    x = torch.randn((m, k), generator=gen, device=DEV, dtype=torch.bfloat16)
    return x, torch.randn((n, k), generator=gen, device=DEV, dtype=torch.bfloat16)


@pytest.mark.parametrize("config", ["256x192", "192x192"])
@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("layout", ["native", "weight_kmajor", "odd_pitch"])
def test_same_bits_as_the_small_tiles(config, shape, layout):
    from rl_engine.backends.rocm.gemm.det_gemm import mfma_gemm

    m, n, k = shape
    x, w = _operands(shape, m + n)
    want = torch.empty((m, n), device=DEV, dtype=torch.bfloat16)
    mfma_gemm(x, w.t(), out=want, config="64x64")
    # a 64-bit product: one bf16 rounding (2^-9 relative) and fp32 sums of k terms
    ref = x.double() @ w.double().t()
    assert bool(((want.double() - ref).abs() <= 2.0**-8 * ref.abs() + 2.0**-22 * k * 16).all())
    b = w.t()
    if layout == "weight_kmajor":
        b = b.contiguous()
    elif layout == "odd_pitch":
        wide = torch.zeros((n, k + 3), device=DEV, dtype=torch.bfloat16)
        wide[:, :k] = w
        b = wide[:, :k].t()
    pad = torch.full((m + 1, n + 8), 7.0, device=DEV, dtype=torch.bfloat16)
    mfma_gemm(x, b, out=pad[:m, :n], config=config)
    assert torch.equal(pad[:m, :n].contiguous().view(torch.int16), want.view(torch.int16))
    assert bool((pad[m] == 7.0).all()) and bool((pad[:, n:] == 7.0).all())


@pytest.mark.parametrize("config", ["256x192", "192x192"])
def test_fp32_results(config):
    from rl_engine import _C, _lib

    x, w = _operands((385, 520, 192), 5)
    got, want = (torch.empty((385, 520), device=DEV, dtype=torch.float32) for _ in range(2))
    _C.gemm_strided(x, w.t(), got, config=_lib.GEMM_CONFIGS[config])
    _C.gemm_strided(x, w.t(), want, config=_lib.GEMM_CONFIGS["64x64"])
    assert torch.equal(got, want)


@pytest.mark.parametrize("tokens,inter", [(360, 12288), (382, 12280), (700, 6144)])
def test_gated_projection_with_192_token_tiles(tokens, inter):
    """Sizes where the fused gate/up runs 192-token tiles: the projection followed by the activation, bit for bit."""
    from rl_engine import _C

    gen = torch.Generator(device=DEV).manual_seed(tokens)
    x = torch.randn((tokens, 256), generator=gen, device=DEV, dtype=torch.bfloat16)
    w = torch.randn((2 * inter, 256), generator=gen, device=DEV, dtype=torch.bfloat16).mul_(0.1)
    y = _C.det_gemm_swiglu(x, w)
    gate_up = torch.empty((tokens, 2 * inter), device=DEV, dtype=torch.bfloat16)
    _C.gemm_strided(x, w.t(), gate_up)
    assert torch.equal(y.view(torch.int16), _C.swiglu_packed_forward(gate_up).view(torch.int16))
