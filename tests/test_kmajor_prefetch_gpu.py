"""The small K-major tiles whose weight panel a ninth wave prefetches: the bits of the plain kernels at every edge."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda"


# features: one panel, panels split between XCDs, a last panel that is not whole; tokens: one reader (no prefetch), two
# with a nearly empty and with a half full second tile, many; reductions: the shortest the ring takes (as many K tiles
# as it holds: no prefetch reaches past the end), one stage more, lengths that end inside a burst of four K tiles
@pytest.mark.parametrize("config,ring", [("64x64", 8), ("128x64", 6), ("128x128", 4)])
@pytest.mark.parametrize("features", [128, 1000, 2056])
@pytest.mark.parametrize("tokens", [40, 67, 104, 128, 200, 700])
def test_prefetched_panels_give_the_same_bits(config, ring, features, tokens):
    from rl_engine import _C, _lib

    gen = torch.Generator(device=DEV).manual_seed(features + tokens)
    code = _lib.GEMM_CONFIGS[config]
    for k_tiles in (ring, ring + 2, ring + 8, 26):
        k = 64 * k_tiles
        x = torch.randn((tokens, k), generator=gen, device=DEV).to(torch.bfloat16)
        w = (0.1 * torch.randn((k, features), generator=gen, device=DEV)).to(torch.bfloat16)
        for dtype in (torch.bfloat16, torch.float32):
            out = torch.empty((tokens, features), dtype=dtype, device=DEV)
            want = torch.empty_like(out)
            _C.gemm_strided(x, w, out, config=code)
            _C.gemm_strided(x, w.t().contiguous().t(), want)  # reduction-contiguous weight: another loop altogether
            bits = torch.int16 if dtype == torch.bfloat16 else torch.int32
            assert torch.equal(out.view(bits), want.view(bits)), (k_tiles, dtype)
