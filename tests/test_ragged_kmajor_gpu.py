"""Reductions that no stage of the small K-major tiles divides: the bits of the other loops."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda"


# reductions around the ring of the small K-major tiles (8 / 6 / 4 K tiles): shorter, exactly one, a part of a stage and a
# part of a K tile behind it, whole chunks only
@pytest.mark.parametrize("config,ring", [("64x64", 8), ("128x64", 6), ("128x128", 4)])
@pytest.mark.parametrize("tokens", [40, 200])
def test_ragged_reductions_of_small_kmajor_tiles(config, ring, tokens):
    from rl_engine import _C, _lib

    gen = torch.Generator(device=DEV).manual_seed(ring + tokens)
    for k in (64 * ring - 8, 64 * ring, 64 * ring + 8, 64 * ring + 64, 64 * ring + 120, 64 * (ring + 7) + 16):
        x = torch.randn((tokens, k), generator=gen, device=DEV).to(torch.bfloat16)
        w = (0.1 * torch.randn((k, 1000), generator=gen, device=DEV)).to(torch.bfloat16)
        out = torch.empty((tokens, 1000), dtype=torch.float32, device=DEV)
        want = torch.empty_like(out)
        _C.gemm_strided(x, w, out, config=_lib.GEMM_CONFIGS[config])
        _C.gemm_strided(x, w.t().contiguous().t(), want)
        assert torch.equal(out.view(torch.int32), want.view(torch.int32)), k
