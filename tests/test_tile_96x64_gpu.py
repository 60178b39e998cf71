"""The 96 x 64 tile of four waves: the bits of the one-wave tile at every edge, the sizes it is chosen for, and the 128 x 64
tile of eight waves where it is not."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda"


@pytest.mark.parametrize("tokens", [1, 31, 64, 65, 127, 193])
@pytest.mark.parametrize("features", [40, 95, 96, 97, 200])
def test_same_bits_as_the_one_wave_tile(tokens, features):
    from rl_engine import _C, _lib

    gen = torch.Generator(device=DEV).manual_seed(tokens * 1000 + features)
    for tiles in (2, 6, 8, 14):  # K tiles: fewer than the seven stages, as many, more
        x = torch.randn((tokens, 64 * tiles), generator=gen, device=DEV, dtype=torch.bfloat16)
        w = torch.randn((features, 64 * tiles), generator=gen, device=DEV, dtype=torch.bfloat16)
        for dtype in (torch.bfloat16, torch.float32):
            pad = torch.full((tokens + 1, features + 8), 7.0, dtype=dtype, device=DEV)
            want = torch.empty((tokens, features), dtype=dtype, device=DEV)
            _C.gemm_strided(x, w.t(), pad[:tokens, :features], config=_lib.GEMM_CONFIGS["96x64_deep"])
            _C.gemm_strided(x, w.t(), want, config=_lib.GEMM_CONFIGS["16x16"])
            bits = torch.int16 if dtype == torch.bfloat16 else torch.int32
            assert torch.equal(pad[:tokens, :features].contiguous().view(bits), want.view(bits)), (tiles, dtype)
            assert bool((pad[tokens] == 7.0).all()) and bool((pad[:, features:] == 7.0).all())


# one token tile of a weight read past the caches, two (96 x 64 and, with more outputs, 128 x 64), three and four
@pytest.mark.parametrize(
    "config,tokens,features,k",
    [("96x64_deep", 50, 24576, 4096), ("96x64_deep", 64, 24500, 1024), ("96x64_deep", 100, 12288, 1024),
     ("128x64_deep", 100, 14336, 1024), ("96x64_deep", 150, 8160, 1152), ("96x64_deep", 192, 6100, 1152), ("96x64_deep", 256, 6144, 4096)],
)  # fmt: skip
def test_chosen_shapes(config, tokens, features, k):
    from rl_engine import _C, _lib

    assert _C.det_gemm_pick_config(tokens, features, k) == _lib.GEMM_CONFIGS[config]
    gen = torch.Generator(device=DEV).manual_seed(tokens)
    x = torch.randn((tokens, k), generator=gen, device=DEV, dtype=torch.bfloat16)
    w = torch.randn((features, k), generator=gen, device=DEV, dtype=torch.bfloat16)
    out, want = (torch.empty((tokens, features), dtype=torch.bfloat16, device=DEV) for _ in range(2))
    _C.gemm_strided(x, w.t(), out)
    _C.gemm_strided(x, w.t(), want, config=_lib.GEMM_CONFIGS["16x16"])
    assert torch.equal(out.view(torch.int16), want.view(torch.int16))
