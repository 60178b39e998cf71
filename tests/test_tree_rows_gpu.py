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


# leaves of 20 and 28, five levels to ten; one row and column, edges of tiles, 16 and 32 rows per wave
@pytest.mark.parametrize("shape", [(1, 1, 640), (2, 4096, 14336), (17, 130, 896), (33, 8200, 1792), (16, 9000, 5120), (300, 4100, 14336),
                                   (70, 16390, 2560), (5, 70, 20480), (40, 16384, 28672)])  # fmt: skip
@pytest.mark.parametrize("special", [False, True])
def test_leaves_that_do_not_start_on_sixteen_bytes(oracle, shape, special):
    test_rows_per_wave_keep_the_bits(oracle, shape, special)


def test_operands_of_other_pitches_and_places(oracle):
    """Rows inside longer ones and repeated rows, whose ends the loads must not pass; a place that is not aligned goes the other way."""
    from rl_engine import _C

    m, n, k = 21, 70, 1792
    gen = torch.Generator(device="cuda").manual_seed(4)
    store = torch.randn(n * (k + 24) + 8, generator=gen, device="cuda", dtype=torch.bfloat16)
    a = torch.randn(m, k, generator=gen, device="cuda", dtype=torch.bfloat16)
    for first, pitch in ((0, k + 24), (0, k), (8, k), (0, 0), (3, k)):
        w = store.as_strided((n, k), (pitch, 1), first)
        for rows in (a, a[:1].expand(m, k)):
            got, want = (torch.empty(m, n, device="cuda", dtype=torch.bfloat16) for _ in range(2))
            _C.gemm_tree_strided(rows, w.t(), got)
            _C.gemm_tree_strided(rows, w.t(), want, 1)
            assert torch.equal(got.view(torch.int16), want.view(torch.int16)), (first, pitch)
