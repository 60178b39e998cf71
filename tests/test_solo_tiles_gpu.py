"""The 256 x 256 tiles with one wave per SIMD at their edges: the bits of the small tiles, nothing written beside the result, one
tile and several of a workgroup (more tiles than compute units), from one K tile on; the fused gate/up on the same loop."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda"
# (tokens, outputs, K): one token, a tile, one more of either, one K tile, two, more tiles than CUs (340, 612), a long reduction
SHAPES = [(1, 8, 64), (256, 256, 64), (257, 255, 128), (128, 384, 192), (300, 777, 4096), (4900, 4200, 64), (9000, 4352, 448)]


def _operands(shape, seed):
    m, n, k = shape
    gen = torch.Generator(device=DEV).manual_seed(seed)
    x = torch.randn((m, k), generator=gen, device=DEV, dtype=torch.bfloat16)
    return x, torch.randn((n, k), generator=gen, device=DEV, dtype=torch.bfloat16)


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("pitch", [8, 3, 0])  # of the result beyond its columns: whole 16-byte stores, element stores
def test_same_bits_as_the_small_tiles(shape, pitch):
    from rl_engine.backends.rocm.gemm.det_gemm import mfma_gemm

    m, n, _ = shape
    x, w = _operands(shape, m + n)
    want = torch.empty((m, n), device=DEV, dtype=torch.bfloat16)
    mfma_gemm(x, w.t(), out=want, config="64x64")
    pad = torch.full((m + 1, n + pitch), 7.0, device=DEV, dtype=torch.bfloat16)
    for _ in range(2):
        mfma_gemm(x, w.t(), out=pad[:m, :n], config="256x256_solo")
        assert torch.equal(pad[:m, :n].contiguous().view(torch.int16), want.view(torch.int16))
    assert bool((pad[m] == 7.0).all()) and bool((pad[:, n:] == 7.0).all())


@pytest.mark.parametrize("shape", [(4096, 4096, 256), (4100, 4300, 64), (9000, 4096, 128)])
def test_the_automatic_choice_runs_them_and_gives_the_bits_of_the_other_loop(shape):
    from rl_engine import _C, _lib

    m, n, k = shape
    pingpong = _lib.GEMM_CONFIGS["256x256"]
    if shape == (4096, 4096, 256):
        assert _C.det_gemm_pick_config(m, n, k) == pingpong  # the shape; how it runs is the launch's choice
    x, w = _operands(shape, 3)
    a, b = (torch.empty((m, n), device=DEV, dtype=torch.bfloat16) for _ in range(2))
    _C.gemm_strided(x, w.t(), a)
    _C.gemm_strided(x, w.t(), b, config=pingpong)
    assert torch.equal(a.view(torch.int16), b.view(torch.int16))


@pytest.mark.parametrize("tokens,inter,k", [(3000, 2040, 64), (4096, 4096, 192), (8190, 2049, 128)])
def test_gated_projection(tokens, inter, k):
    """Sizes where the fused gate/up runs them: the projection followed by the activation, bit for bit."""
    from rl_engine import _C

    gen = torch.Generator(device=DEV).manual_seed(tokens)
    x = torch.randn((tokens, k), generator=gen, device=DEV, dtype=torch.bfloat16)
    w = torch.randn((2 * inter, k), generator=gen, device=DEV, dtype=torch.bfloat16).mul_(0.1)
    y = _C.det_gemm_swiglu(x, w)
    gate_up = torch.empty((tokens, 2 * inter), device=DEV, dtype=torch.bfloat16)
    _C.gemm_strided(x, w.t(), gate_up, config=3)  # 128 x 128
    assert torch.equal(y.view(torch.int16), _C.swiglu_packed_forward(gate_up).view(torch.int16))
