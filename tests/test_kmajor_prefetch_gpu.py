"""The small K-major tiles whose weight panel a ninth wave prefetches: the bits of the plain kernels at every edge."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda"


def _same_bits(code, features, tokens, k_tiles, gen):
    from rl_engine import _C

    k = 64 * k_tiles
    x = torch.randn((tokens, k), generator=gen, device=DEV, dtype=torch.bfloat16)
    w = torch.randn((k, features), generator=gen, device=DEV, dtype=torch.bfloat16).mul_(0.1)
    for dtype in (torch.bfloat16, torch.float32):
        out = torch.empty((tokens, features), dtype=dtype, device=DEV)
        want = torch.empty_like(out)
        _C.gemm_strided(x, w, out, config=code)
        _C.gemm_strided(x, w.t().contiguous().t(), want)  # reduction-contiguous weight: another loop altogether
        bits = torch.int16 if dtype == torch.bfloat16 else torch.int32
        assert torch.equal(out.view(bits), want.view(bits)), (k_tiles, dtype)


# The ring at its shortest reduction (as many K tiles as it holds), one stage more, and longer ones.
@pytest.mark.parametrize("config,ring", [("64x64", 8), ("128x64", 6), ("128x128", 4)])
@pytest.mark.parametrize("features", [128, 1000, 2056])
@pytest.mark.parametrize("tokens", [40, 67, 104, 128, 200, 700])
def test_short_reductions_give_the_same_bits(config, ring, features, tokens):
    from rl_engine import _lib

    gen = torch.Generator(device=DEV).manual_seed(features + tokens)
    for k_tiles in (ring, ring + 2, ring + 8, 26):
        _same_bits(_lib.GEMM_CONFIGS[config], features, tokens, k_tiles, gen)


# Weights of 128 MiB run with the ninth wave. features: one panel, panels split between XCDs, a last panel that is not
# whole; tokens: one reader (no prefetch), two with a nearly empty and with a half full second tile, many; reductions that
# end with a whole burst of four K tiles and inside one.
@pytest.mark.parametrize("config", ["64x64", "128x64", "128x128"])
@pytest.mark.parametrize("features", [128, 1000, 2056])
@pytest.mark.parametrize("tokens", [40, 67, 104, 128, 200, 700])
def test_prefetched_panels_give_the_same_bits(config, features, tokens):
    from rl_engine import _lib

    gen = torch.Generator(device=DEV).manual_seed(features + tokens)
    k_tiles = -(-(1 << 26) // (64 * features)) + 3 & ~3
    for extra in (0, 2):
        _same_bits(_lib.GEMM_CONFIGS[config], features, tokens, k_tiles + extra, gen)
