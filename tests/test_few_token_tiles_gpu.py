"""The tiles of four waves (32 x 32 to 64 x 160): the bits of the other kernels at every edge."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda"


# tokens: below, at and above the edges of the tiles, and of the one and a half tiles that bring in the prefetching wave;
# features: less than a tile, whole tiles, a last tile that is not whole; reductions: the fewest stages, fewer stages than the ring holds, more
@pytest.mark.parametrize("config,stage", [("32x32_deep", 128), ("32x64_deep", 256), ("64x32_deep", 256), ("64x96_deep", 128), ("64x160_deep", 128),
                                          ("128x64_deep", 128)])
@pytest.mark.parametrize("tokens", [1, 31, 32, 33, 65, 95, 96, 97, 129, 144, 145, 160, 161, 193, 241])
@pytest.mark.parametrize("features", [40, 64, 200])
def test_same_bits_as_the_one_wave_tile(config, stage, tokens, features):
    from rl_engine import _C, _lib

    gen = torch.Generator(device=DEV).manual_seed(tokens * 1000 + features)
    for stages in (1, 2, 3, 7):
        k = stage * stages
        x = torch.randn((tokens, k), generator=gen, device=DEV, dtype=torch.bfloat16)
        w = torch.randn((features, k), generator=gen, device=DEV, dtype=torch.bfloat16)
        for dtype in (torch.bfloat16, torch.float32):
            out = torch.full((tokens, features), 7.0, dtype=dtype, device=DEV)
            want = torch.empty_like(out)
            _C.gemm_strided(x, w.t(), out, config=_lib.GEMM_CONFIGS[config])
            _C.gemm_strided(x, w.t(), want, config=_lib.GEMM_CONFIGS["16x16"])
            bits = torch.int16 if dtype == torch.bfloat16 else torch.int32
            assert torch.equal(out.view(bits), want.view(bits)), (stages, dtype)


# Shapes that the automatic choice gives to them, with a padded row pitch, for every form that it reaches: the plain loop,
# the weight read past the caches (one token tile, from 96 MiB of weight), the prefetching wave (several token tiles: from
# 96 MiB and with the last tile more than half full for 32 x 64 and 64 x 32, else always); each with a ragged neighbour
# (a last tile that is not whole, an odd number of stages).
@pytest.mark.parametrize(
    "config,tokens,features,k",
    [("32x32_deep", 20, 6144, 4096), ("32x32_deep", 50, 4096, 4096), ("32x32_deep", 30, 6144, 8320),
     ("32x64_deep", 65, 4096, 4096), ("32x64_deep", 200, 1536, 4096), ("32x64_deep", 80, 4096, 12288),
     ("32x64_deep", 64, 8192, 8192), ("32x64_deep", 61, 8190, 8448), ("32x64_deep", 128, 4096, 12544), ("32x64_deep", 101, 4090, 12544),
     ("64x32_deep", 20, 9000, 1280), ("64x32_deep", 20, 12288, 4096), ("64x32_deep", 66, 5120, 25600),
     ("64x32_deep", 96, 5120, 25600), ("64x32_deep", 85, 5118, 25856),
     ("64x96_deep", 140, 8190, 1152), ("64x96_deep", 90, 12288, 4096), ("64x96_deep", 333, 4096, 12288), ("64x96_deep", 150, 8190, 1152),
     ("64x160_deep", 150, 12288, 2048), ("64x160_deep", 150, 12288, 4096), ("64x160_deep", 129, 12346, 4224),
     ("64x160_deep", 600, 4096, 4096), ("64x160_deep", 651, 3250, 4224),
     ("128x64_deep", 500, 4096, 4096), ("128x64_deep", 120, 14336, 4096), ("128x64_deep", 97, 16380, 1152),
     ("96x64_deep", 120, 12288, 4096)],
)  # fmt: skip
def test_chosen_shapes(config, tokens, features, k):
    from rl_engine import _C, _lib

    assert _C.det_gemm_pick_config(tokens, features, k) == _lib.GEMM_CONFIGS[config]
    gen = torch.Generator(device=DEV).manual_seed(tokens)
    x = torch.randn((tokens, k + 8), generator=gen, device=DEV, dtype=torch.bfloat16)[:, :k]
    w = torch.randn((features, k), generator=gen, device=DEV, dtype=torch.bfloat16)
    out = torch.empty((tokens, features), dtype=torch.bfloat16, device=DEV)
    want = torch.empty_like(out)
    _C.gemm_strided(x, w.t(), out)
    _C.gemm_strided(x, w.t(), want, config=_lib.GEMM_CONFIGS["16x16"])
    assert torch.equal(out.view(torch.int16), want.view(torch.int16))
