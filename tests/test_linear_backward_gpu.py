"""Both gradients of a linear layer in one launch (csrc/det_gemm_pair.hip): the bits of two launches at the edges of its
tiles, in every configuration and operand form, and nothing written beside the results."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda"
CONFIGS = range(2, 9)  # rlk_linear_bwd_config: every one-launch configuration
# (tokens, inputs, outputs): one tile and less, a token more than a tile of each height, ragged everything, reductions of
# dX that no stage divides, many tiles of one product beside few of the other, both orders of the two
SHAPES = [
    (1, 8, 8), (64, 64, 64), (65, 136, 200), (129, 264, 328), (257, 512, 72), (300, 1032, 2056),
    (1000, 8, 4104), (130, 4104, 16), (2047, 1000, 1024), (520, 264, 12296),
]  # fmt: skip


def _rand(gen, *shape):
    return torch.randn(shape, generator=gen, device=DEV, dtype=torch.bfloat16)


def _backward(g, x, w, config, dx_pitch=0, dw_pitch=0):
    """dx and dw inside guarded buffers, which stay as they were around the results."""
    from rl_engine import _lib

    (m, n), k = g.shape, x.size(1)
    dx = torch.full((m + 1, k + dx_pitch), 7.0, device=DEV, dtype=torch.bfloat16)
    dw = torch.full((n + 1, k + dw_pitch), 7.0, device=DEV, dtype=torch.bfloat16)
    status = _lib.load().rlk_linear_bwd_bf16(
        g.data_ptr(), g.stride(0), x.data_ptr(), x.stride(0), w.data_ptr(), w.stride(0), dx.data_ptr(), dx.stride(0),
        dw.data_ptr(), dw.stride(0), m, k, n, config, torch.cuda.current_stream().cuda_stream,
    )  # fmt: skip
    _lib.check(status, "rlk_linear_bwd_bf16 failed")
    for t, rows in ((dx, m), (dw, n)):
        assert bool((t[rows] == 7.0).all()) and bool((t[:, k:] == 7.0).all())
    return dx[:m, :k].contiguous().view(torch.int16), dw[:n, :k].contiguous().view(torch.int16)


@pytest.mark.parametrize("shape", SHAPES)
def test_one_launch_gives_the_bits_of_two(shape):
    m, k, n = shape
    gen = torch.Generator(device=DEV).manual_seed(m + n)
    g, x, w = _rand(gen, m, n), _rand(gen, m, k), _rand(gen, n, k)
    want_dx, want_dw = _backward(g, x, w, 1)
    ref_dx, ref_dw = g.double() @ w.double(), g.double().t() @ x.double()
    # one bf16 rounding (2^-9 relative) and fp32 sums of at most max(m, n) terms around the 64-bit products
    for got, ref, terms in ((want_dx, ref_dx, n), (want_dw, ref_dw, m)):
        err = (got.view(torch.bfloat16).double() - ref).abs()
        assert bool((err <= 2.0**-8 * ref.abs() + 2.0**-22 * terms * 16).all())
    for config in CONFIGS:
        dx, dw = _backward(g, x, w, config, dx_pitch=8, dw_pitch=16)
        assert torch.equal(dx, want_dx) and torch.equal(dw, want_dw), config
    dx, dw = _backward(g, x, w, 0)
    assert torch.equal(dx, want_dx) and torch.equal(dw, want_dw)


@pytest.mark.parametrize("form", ["plain", "pitch", "odd_pitch", "offset", "transposed", "one_row_repeated"])
@pytest.mark.parametrize("operand", ["grad", "other"])
@pytest.mark.parametrize("tokens,inputs,outputs", [(67, 136, 200), (300, 264, 1032), (70, 100, 72)])
def test_gradients_of_every_operand_form(form, operand, tokens, inputs, outputs):
    from rl_engine import _C
    from rl_engine.backends.rocm.gemm import det_gemm
    from test_linear_gradient_paths_gpu import _form

    gen = torch.Generator(device=DEV).manual_seed(tokens)
    x, w, g = _rand(gen, tokens, inputs), _rand(gen, outputs, inputs), _rand(gen, tokens, outputs)
    if operand == "grad":
        g = _form(g, form)
    else:
        x, w = _form(x, form), _form(w, form)
    dx, dw = det_gemm.mfma_linear_gradients(x, w, g)
    want_dx, want_dw = torch.empty_like(dx), torch.empty_like(dw)
    _C.gemm_strided(g.contiguous(), w.t().contiguous().t(), want_dx)
    _C.gemm_strided(g.t().contiguous(), x.t().contiguous().t(), want_dw)
    assert torch.equal(dx.view(torch.int16), want_dx.view(torch.int16))
    assert torch.equal(dw.view(torch.int16), want_dw.view(torch.int16))


REST_BESIDE = 0x100  # RLK_LINEAR_BWD_CFG_REST_BESIDE


@pytest.mark.parametrize("config", CONFIGS)
@pytest.mark.parametrize("tokens", [257, 280, 576, 577, 1279])  # rests of 1, 24, 64, 65 and 255 behind one, two and four tiles
def test_the_rest_of_dx_beside_dw(config, tokens):
    """dX in two parts, the second in the launch of dW: operands and results with pitches of their own."""
    k, n = 264, 1032
    gen = torch.Generator(device=DEV).manual_seed(tokens)
    g, x, w = (_rand(gen, rows, cols + pad)[:, :cols] for rows, cols, pad in ((tokens, n, 8), (tokens, k, 24), (n, k, 16)))
    want = _backward(g, x, w, 1)
    got = _backward(g, x, w, config | REST_BESIDE, dx_pitch=8, dw_pitch=16)
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])


@pytest.mark.parametrize("tokens,inputs,outputs", [(193, 1024, 6144), (256, 1032, 2056), (300, 264, 1032), (4120, 1024, 4096)])
def test_one_of_many_weights(tokens, inputs, outputs):
    """The choice for weights that come from HBM again: the same bits."""
    from rl_engine import _lib

    gen = torch.Generator(device=DEV).manual_seed(tokens)
    g, x, w = _rand(gen, tokens, outputs), _rand(gen, tokens, inputs), _rand(gen, outputs, inputs)
    want = _backward(g, x, w, 1)
    got = _backward(g, x, w, _lib.LINEAR_BWD_MANY_WEIGHTS)
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])


@pytest.mark.parametrize("tokens", [4097, 4120, 4160, 4161])
def test_few_tokens_behind_whole_tiles(tokens):
    """A token count just above whole tiles: up to 64 tokens beside dW, by the automatic choice."""
    from rl_engine import _lib

    k = n = 4096
    lib = _lib.load()
    assert bool(lib.rlk_linear_bwd_pick_config(tokens, k, n, 0) & REST_BESIDE) == (tokens <= 4160)
    gen = torch.Generator(device=DEV).manual_seed(tokens)
    g, x, w = _rand(gen, tokens, n), _rand(gen, tokens, k), _rand(gen, n, k)
    want = _backward(g, x, w, 1)
    got = _backward(g, x, w, 0)
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])


@pytest.mark.parametrize("tokens", [4097, 4120, 4160])
@pytest.mark.parametrize("vocab", [4093, 4096])
def test_few_tokens_behind_whole_tiles_in_the_logp_backward(tokens, vocab):
    """The same in the LogP backward, whose d(logits) rows go on to a whole chunk behind the vocabulary: the bits of each
    gradient asked for alone."""
    from rl_engine import _C, _lib

    assert _lib.load().rlk_linear_bwd_pick_config(tokens, 4096, vocab, 1) & REST_BESIDE
    gen = torch.Generator(device=DEV).manual_seed(tokens)
    h, w = _rand(gen, tokens, 4096), _rand(gen, vocab, 4096).mul_(0.02)
    ids = torch.randint(0, vocab, (tokens,), generator=gen, device=DEV)
    _, lse = _C.fused_linear_logp(h, w, ids)
    g = torch.randn((tokens,), generator=gen, device=DEV)
    both = _C.fused_linear_logp_bwd(h, w, ids, lse, g, None)
    hidden = _C.fused_linear_logp_bwd(h, w, ids, lse, g, None, need_grad_weight=False)
    weight = _C.fused_linear_logp_bwd(h, w, ids, lse, g, None, need_grad_hidden=False)
    assert torch.equal(both[0].view(torch.int16), hidden[0].view(torch.int16))
    assert torch.equal(both[1].view(torch.int16), weight[1].view(torch.int16))


def test_refused_arguments():
    from rl_engine import _lib

    m, k, n = 8, 8, 16
    gen = torch.Generator(device=DEV).manual_seed(1)
    g, x, w = _rand(gen, m, n), _rand(gen, m, k), _rand(gen, n, k)
    dx, dw = torch.empty_like(x), torch.empty_like(w)
    lib = _lib.load()

    def call(grad, config):
        return lib.rlk_linear_bwd_bf16(grad, n, x.data_ptr(), k, w.data_ptr(), k, dx.data_ptr(), k, dw.data_ptr(), k, m, k, n, config, None)

    assert call(None, 0) < 0
    for config in (-1, 9, REST_BESIDE, REST_BESIDE | 1, REST_BESIDE | 9, 2 * REST_BESIDE, 0x401, 0x500):
        assert call(g.data_ptr(), config) < 0, config


def test_a_captured_backward_replays():
    """Two gradients under HIP-graph capture: every replay gives the eager bits on the inputs of that replay."""
    from rl_engine.backends.rocm.gemm import det_gemm

    gen = torch.Generator(device=DEV).manual_seed(3)
    x, w, g = _rand(gen, 300, 512), _rand(gen, 1024, 512), _rand(gen, 300, 1024)
    det_gemm.mfma_linear_gradients(x, w, g)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        dx, dw = det_gemm.mfma_linear_gradients(x, w, g)
    for _ in range(3):
        g.copy_(_rand(gen, 300, 1024))
        graph.replay()
        want_dx, want_dw = det_gemm.mfma_linear_input_gradient(g, w), det_gemm.mfma_linear_weight_gradient(x, g)
        torch.cuda.synchronize()
        assert torch.equal(dx.view(torch.int16), want_dx.view(torch.int16))
        assert torch.equal(dw.view(torch.int16), want_dw.view(torch.int16))
