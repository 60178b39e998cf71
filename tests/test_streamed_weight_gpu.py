"""Weights of 96 MiB and more are read past the caches where one token tile reads them, of 128 MiB where two do: the same bits."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda"
N, K = 16386, 4096  # 128.02 MiB, and 2 rows more than whole tiles


@pytest.fixture(scope="module")
def operands():
    gen = torch.Generator(device=DEV).manual_seed(90)
    w = torch.randn((N, K), generator=gen, device=DEV).to(torch.bfloat16) * 0.02
    x = torch.randn((300, K), generator=gen, device=DEV).to(torch.bfloat16)
    return x, w


# one token, the last of the 16-token panel, one and two whole token tiles of every height, the sizes beside them
@pytest.mark.parametrize("tokens", [1, 16, 17, 64, 65, 127, 128, 129, 255, 256, 257])
def test_gemm_rows_equal_those_of_a_small_weight(operands, tokens):
    from rl_engine import _C

    x, w = operands
    out = _C.det_gemm_fwd_rhs_transposed(x[:tokens], w)
    for lo, hi in ((0, 130), (6100, 6300), (N - 131, N)):  # 131 rows are 1 MiB: the ordinary loads
        part = _C.det_gemm_fwd_rhs_transposed(x[:tokens], w[lo:hi])
        assert torch.equal(out[:, lo:hi].view(torch.int16), part.view(torch.int16))


# up to 128 tokens in tiles of 16, 32, 48 and 64 features: weights of 96 to 194 MiB
@pytest.mark.parametrize("tokens", [1, 16, 17, 63, 64, 65, 96, 97, 128, 129, 256, 257])
@pytest.mark.parametrize("rows,k", [(8190, 6272), (16384, 4096), (N, 4096), (24800, 4096)])
def test_gated_projection_equals_gemm_and_activation(operands, tokens, rows, k):
    from rl_engine import _C
    from rl_engine.backends.rocm.gemm import swiglu_gemm

    x, w = (t.flatten()[: n * k].view(n, k) if t.numel() >= n * k else t.flatten().repeat(2)[: n * k].view(n, k)
            for t, n in zip(operands, (tokens, rows)))  # fmt: skip
    fused = swiglu_gemm.forward(x, w)
    two = _C.swiglu_packed_forward(_C.det_gemm_fwd_rhs_transposed(x, w))
    assert torch.equal(fused.view(torch.int16), two.view(torch.int16))


@pytest.mark.parametrize("tokens", [1, 63, 64, 65, 128, 129])
def test_logp_rows_equal_those_of_a_larger_batch(operands, tokens):
    from rl_engine.ops.logprob import deterministic_linear_logp

    x, w = operands
    ids = (torch.arange(300, device=DEV) * 41) % N
    with torch.no_grad():
        whole = deterministic_linear_logp(x, w, ids)
        part = deterministic_linear_logp(x[:tokens], w, ids[:tokens])
    for a, b in zip(whole, part):
        assert torch.equal(a[:tokens].view(torch.int32), b.view(torch.int32))
