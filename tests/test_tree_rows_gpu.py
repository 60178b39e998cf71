"""The k-tree kernel with 16 and with 32 rows per wave (csrc/det_gemm_tree.hip: det_gemm_tree_rows_kernel) at the edges of
its tiles, trees and choice: bit-exact against the oracle on the columns it can afford, and against the one-fma-per-term
kernel of the library everywhere."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import inputs

pytestmark = pytest.mark.gpu

# (M, N, K): 16 rows per wave - one row more than the tile, ragged columns, five levels, leaves of 24 and 32, the deepest
# tree - then four levels (always 32 rows), then grids large enough for 32 rows per wave
SHAPES = [
    (17, 8200, 1024), (50, 4100, 3072), (33, 4096, 12288), (16, 9000, 768), (17, 8256, 32768),
    (5, 100, 384), (33, 130, 512),
    (64, 16383, 1024), (33, 32800, 768), (200, 6150, 4096), (256, 4096, 12288),
]  # fmt: skip


def _special(t: torch.Tensor, seed: int) -> torch.Tensor:
    """Zeros of both signs, bf16 denormals, the largest values, infinities and NaN in a few rows."""
    gen = torch.Generator(device=t.device).manual_seed(seed)
    values = [0.0, -0.0, 1e-39, -3e-40, 3.3e38, -3.3e38, float("inf"), float("-inf"), float("nan")]
    flat = t.view(-1)
    for i, v in enumerate(values):
        count = max(2, t.numel() // 4000) if i < 4 else 2
        flat[torch.randint(0, flat.numel(), (count,), generator=gen, device=t.device)] = v
    return t


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("special", [False, True])
def test_rows_per_wave_keep_the_bits(oracle, shape, special):
    from rl_engine import _C
    from rl_engine.backends.rocm.gemm.det_gemm import tree_gemm

    m, n, k = shape
    gen = torch.Generator(device="cuda").manual_seed(k + n)
    a = torch.randn(m, k, generator=gen, device="cuda", dtype=torch.bfloat16)
    w = torch.randn(n, k, generator=gen, device="cuda", dtype=torch.bfloat16).mul_(0.02)
    if special:
        _special(a, 1), _special(w, 2)
    pad = torch.full((m + 1, n + 8), 7.0, device="cuda", dtype=torch.bfloat16)  # nothing behind the result is written
    out = pad[:m, :n]
    tree_gemm(a, w.t(), out=out)
    assert bool((pad[m] == 7.0).all()) and bool((pad[:, n:] == 7.0).all())
    by_term = torch.empty(m, n, device="cuda", dtype=torch.bfloat16)
    _C.gemm_tree_strided(a, w.t(), by_term, 1)
    nan = torch.isnan(by_term)
    assert torch.equal(torch.isnan(out), nan)
    assert torch.equal(torch.where(nan, 0, out.contiguous().view(torch.int16)), torch.where(nan, 0, by_term.view(torch.int16)))
    if not special:
        columns = torch.tensor(sorted({0, 15, 16, 63, 64, n // 2, n - 1} & set(range(n))), device="cuda")
        want = oracle.k_tree_gemm(inputs.bits(a.cpu()), inputs.bits(w[columns].cpu()))
        assert np.array_equal(inputs.bits(out[:, columns].contiguous().cpu()), want)
