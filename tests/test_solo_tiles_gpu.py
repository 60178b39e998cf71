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


# sizes that the choice gives each of the gated tiles, on 256 CUs: 64 x 128, 64 x 192, 128 x 128, 192 x 128, 128 x 192, 256 x 128, 192 x
# 192, 192 x 256, 256 x 192; rows of the result whole 16 bytes (whole stores and element stores of the last tile) and not
@pytest.mark.parametrize("tokens,inter", [(129, 3064), (300, 2049), (150, 6136), (411, 3064), (390, 6136), (390, 6141), (947, 3064), (947, 3066),
                                          (640, 6136), (310, 12280), (310, 12281), (474, 12280), (1800, 3064)])  # fmt: skip
@pytest.mark.parametrize("k", [64, 128, 512])
def test_gated_tiles_of_few_tokens(tokens, inter, k):
    """The projection followed by the activation, bit for bit; from one K tile to more than the stages of a ring."""
    from rl_engine import _C

    gen = torch.Generator(device=DEV).manual_seed(tokens + k)
    x = torch.randn((tokens, k), generator=gen, device=DEV, dtype=torch.bfloat16)
    w = torch.randn((2 * inter, k), generator=gen, device=DEV, dtype=torch.bfloat16).mul_(0.1)
    gate_up = torch.empty((tokens, 2 * inter), device=DEV, dtype=torch.bfloat16)
    _C.gemm_strided(x, w.t(), gate_up, config=5)  # 64 x 64
    want = _C.swiglu_packed_forward(gate_up)
    for _ in range(2):
        assert torch.equal(_C.det_gemm_swiglu(x, w).view(torch.int16), want.view(torch.int16))


@pytest.mark.parametrize("tokens,inter,k", [(1, 8, 64), (128, 264, 128), (129, 3064, 64), (300, 2049, 192), (150, 6136, 128), (411, 3064, 512), (390, 6141, 128),
                                            (947, 3064, 64), (640, 6136, 128), (310, 12280, 64), (474, 12280, 128), (1800, 3064, 128),
                                            (4096, 4100, 128), (200, 264, 72)])  # fmt: skip
def test_gate_and_up_of_a_training_step(tokens, inter, k):
    """Two weights, both projections kept: the bits of three launches; what the one launch does not take among the sizes."""
    from rl_engine import _C, _lib

    gen = torch.Generator(device=DEV).manual_seed(tokens + k)
    x = torch.randn((tokens, k), generator=gen, device=DEV, dtype=torch.bfloat16)
    up_w, gate_w = (torch.randn((inter, k), generator=gen, device=DEV, dtype=torch.bfloat16).mul_(0.1) for _ in range(2))
    want = []
    for w in (gate_w, up_w):
        want.append(torch.empty((tokens, inter), device=DEV, dtype=torch.bfloat16))
        _C.gemm_strided(x, w.t(), want[-1], config=5)  # 64 x 64
    want.append(_C.swiglu_forward(*want))
    got = [torch.full((tokens, inter), 7.0, device=DEV, dtype=torch.bfloat16) for _ in range(3)]
    status = _lib.load().rlk_det_gemm_swiglu_training_bf16(
        x.data_ptr(), k, gate_w.data_ptr(), up_w.data_ptr(), k, *(t.data_ptr() for t in got), inter, tokens, inter, k,
        torch.cuda.current_stream().cuda_stream)  # fmt: skip
    assert status == 0
    assert all(torch.equal(g.view(torch.int16), w.view(torch.int16)) for g, w in zip(got, want))


# one K tile, as many as stages and one more or less, edges of tiles of either side, tails of a few rows, more tiles than CUs
@pytest.mark.parametrize("shape", [(1, 8, 64), (192, 192, 128), (129, 200, 192), (400, 392, 256), (257, 777, 320), (300, 500, 1024), (3100, 3200, 448)])
@pytest.mark.parametrize("name", ["256x192", "192x256", "192x192", "256x128", "192x128"])
def test_smaller_shapes_on_four_waves(shape, name):
    """The bits of the small tiles; whole 16-byte stores and element stores, nothing written beside the result."""
    from rl_engine import _C, _lib

    m, n, _ = shape
    x, w = _operands(shape, m * n)
    want = torch.empty((m, n), device=DEV, dtype=torch.bfloat16)
    _C.gemm_strided(x, w.t(), want, config=_lib.GEMM_CONFIGS["64x64"])
    for pitch in (8, 3):
        pad = torch.full((m + 1, n + pitch), 7.0, device=DEV, dtype=torch.bfloat16)
        _C.gemm_strided(x, w.t(), pad[:m, :n], config=_lib.GEMM_CONFIGS[name] | _lib.FOUR_WAVES)
        assert torch.equal(pad[:m, :n].contiguous().view(torch.int16), want.view(torch.int16))
        assert bool((pad[m] == 7.0).all()) and bool((pad[:, n:] == 7.0).all())
    if name in ("256x192", "256x128"):  # a K-major weight, whose rows come in eights
        n8 = (n + 7) // 8 * 8
        wt = torch.zeros((w.size(1), n8), device=DEV, dtype=torch.bfloat16)
        wt[:, :n] = w.t()
        for k in (w.size(1), w.size(1) - 8, w.size(1) - 56):
            _C.gemm_strided(x[:, :k].contiguous(), w[:, :k].contiguous().t(), want, config=_lib.GEMM_CONFIGS["64x64"])
            got = torch.empty((m, n8), device=DEV, dtype=torch.bfloat16)
            _C.gemm_strided(x[:, :k].contiguous(), wt[:k], got, config=_lib.GEMM_CONFIGS[name] | _lib.FOUR_WAVES)
            assert torch.equal(got[:, :n].contiguous().view(torch.int16), want.view(torch.int16)), k


# rows of the result that start on 16, 8, 4 and 2 bytes, by their pitch and by where the first one starts; columns that end inside a
# lane's run, on it and on a span of 64
@pytest.mark.parametrize("outputs", [320, 328, 517, 382])
@pytest.mark.parametrize("pitch,first", [(0, 0), (4, 4), (2, 8), (2, 2), (1, 0), (3, 1), (8, 1)])
@pytest.mark.parametrize("name", ["256x256_solo", "192x256", "192x192", "192x128", "256x192 K-major"])
def test_rows_of_every_alignment(outputs, pitch, first, name):
    """The bits of the small tiles, nothing written before, between and behind the rows."""
    from rl_engine import _C, _lib

    m, n, k = 300, outputs, 128
    x, w = _operands((m, n, k), outputs + pitch)
    want = torch.empty((m, n), device=DEV, dtype=torch.bfloat16)
    _C.gemm_strided(x, w.t(), want, config=_lib.GEMM_CONFIGS["64x64"])
    ld = (n + 7) // 8 * 8 + pitch
    flat = torch.full((first + m * ld + 8,), 7.0, device=DEV, dtype=torch.bfloat16)
    got = flat.as_strided((m, n), (ld, 1), first)
    shape, _, kmajor = name.partition(" ")
    b = w.t()
    if kmajor:
        n8 = (n + 7) // 8 * 8
        wt = torch.zeros((k, n8), device=DEV, dtype=torch.bfloat16)
        wt[:, :n] = w.t()
        if n8 != n:  # a K-major weight has whole eights of outputs
            got = flat.as_strided((m, n8), (ld, 1), first)
            b = wt
            want = torch.cat([want, torch.zeros((m, n8 - n), device=DEV, dtype=torch.bfloat16)], 1)
        else:
            b = w.t().contiguous()
    config = _lib.GEMM_CONFIGS[shape] | (_lib.FOUR_WAVES if "solo" not in shape else 0)
    _C.gemm_strided(x, b, got, config=config)
    assert torch.equal(got.contiguous().view(torch.int16), want.view(torch.int16))
    got.fill_(7.0)
    assert bool((flat == 7.0).all())


# the same of the fused gate/up: whole tiles and ragged ones, rows on 8, 4 and 2 bytes
@pytest.mark.parametrize("inter", [3068, 3070, 3071, 516, 514, 515])
@pytest.mark.parametrize("tokens", [129, 411, 1029, 4100])
def test_gated_rows_of_every_alignment(tokens, inter):
    from rl_engine import _C, _lib

    k = 64
    gen = torch.Generator(device=DEV).manual_seed(tokens + inter)
    x = torch.randn((tokens, k), generator=gen, device=DEV, dtype=torch.bfloat16)
    w = torch.randn((2 * inter, k), generator=gen, device=DEV, dtype=torch.bfloat16).mul_(0.1)
    gate_up = torch.empty((tokens, 2 * inter), device=DEV, dtype=torch.bfloat16)
    _C.gemm_strided(x, w.t(), gate_up, config=5)  # 64 x 64
    want = _C.swiglu_packed_forward(gate_up)
    assert torch.equal(_C.det_gemm_swiglu(x, w).view(torch.int16), want.view(torch.int16))
    got = [torch.full((tokens, inter), 7.0, device=DEV, dtype=torch.bfloat16) for _ in range(3)]
    gate_w, up_w = w[:inter].contiguous(), w[inter:].contiguous()
    assert 0 == _lib.load().rlk_det_gemm_swiglu_training_bf16(
        x.data_ptr(), k, gate_w.data_ptr(), up_w.data_ptr(), k, *(t.data_ptr() for t in got), inter, tokens, inter, k,
        torch.cuda.current_stream().cuda_stream)  # fmt: skip
    for g, part in zip(got, (gate_up[:, :inter], gate_up[:, inter:], want)):
        assert torch.equal(g.view(torch.int16), part.contiguous().view(torch.int16))


# K-major tokens, which the four-wave forms of these shapes do not take: whole K tiles (read as rows of 64 values they would
# be there) and a ragged reduction
@pytest.mark.parametrize("shape", [(264, 520, 64), (520, 392, 200), (256, 384, 256)])
@pytest.mark.parametrize("w_kmajor", [False, True])
@pytest.mark.parametrize("name", ["256x192", "256x128", "192x256", "192x192", "192x128"])
def test_four_waves_asked_for_with_kmajor_tokens_run_the_plain_shape(shape, w_kmajor, name):
    from rl_engine import _C, _lib

    m, n, k = shape
    x, w = _operands(shape, m + n + k)
    want = torch.empty((m, n), device=DEV, dtype=torch.bfloat16)
    _C.gemm_strided(x, w.t(), want, config=_lib.GEMM_CONFIGS["64x64"])
    xt = x.t().contiguous().t()
    b = w.t().contiguous() if w_kmajor else w.t()
    for config in (_lib.GEMM_CONFIGS[name], _lib.GEMM_CONFIGS[name] | _lib.FOUR_WAVES):
        got = torch.full((m, n), 7.0, device=DEV, dtype=torch.bfloat16)
        _C.gemm_strided(xt, b, got, config=config)
        assert torch.equal(got.view(torch.int16), want.view(torch.int16)), config


# (tokens, outputs, K): one K tile and less, a few values more than whole K tiles, odd ones, edges of tiles of either side, more
# tiles than CUs
KMAJOR_SHAPES = [(8, 8, 8), (256, 256, 24), (264, 520, 64), (248, 776, 72), (1000, 264, 200), (512, 512, 2056), (4360, 4360, 136)]


@pytest.mark.parametrize("shape", KMAJOR_SHAPES)
@pytest.mark.parametrize("w_kmajor,x_kmajor", [(True, False), (False, True), (True, True)])
@pytest.mark.parametrize("pitch", [8, 3])  # of the result beyond its columns: whole 16-byte stores, element stores
def test_kmajor_operands(shape, w_kmajor, x_kmajor, pitch):
    """The bits of the two-group loop of the same operands; with both K-major also reductions of odd length."""
    from rl_engine import _C, _lib

    m, n, k = shape
    gen = torch.Generator(device=DEV).manual_seed(m + k)

    def operand(rows, length, kmajor):
        shape = (length, rows) if kmajor else (rows, length)
        t = torch.randn(shape, generator=gen, device=DEV, dtype=torch.bfloat16)
        return t.t() if kmajor else t

    for length in (k, k + 1, k + 63) if w_kmajor and x_kmajor else (k,):
        if not w_kmajor and length % 64 == 0 and x_kmajor:
            length += 8
        x, w = operand(m, length, x_kmajor), operand(n, length, w_kmajor)
        want = torch.empty((m, n), device=DEV, dtype=torch.bfloat16)
        _C.gemm_strided(x.contiguous(), w.contiguous().t(), want, config=3)  # 128 x 128, native operands
        pad = torch.full((m + 1, n + pitch), 7.0, device=DEV, dtype=torch.bfloat16)
        for _ in range(2):
            _C.gemm_strided(x, w.t(), pad[:m, :n], config=_lib.GEMM_CONFIGS["256x256_solo"])
            assert torch.equal(pad[:m, :n].contiguous().view(torch.int16), want.view(torch.int16)), length
        assert bool((pad[m] == 7.0).all()) and bool((pad[:, n:] == 7.0).all())


def test_nothing_past_a_reduction_is_used():
    """The values behind the reduction's end, which lie in memory beside it, are NaN: the next K rows of K-major operands, the rest
    of the rows of a native one."""
    from rl_engine import _C, _lib

    m, n, k = 520, 264, 136
    x = torch.full((m, k + 64), float("nan"), device=DEV, dtype=torch.bfloat16)
    xt = torch.full((k + 64, m), float("nan"), device=DEV, dtype=torch.bfloat16)
    w = torch.full((k + 64, n), float("nan"), device=DEV, dtype=torch.bfloat16)
    x[:, :k].normal_()
    xt[:k] = x[:, :k].t()
    w[:k].normal_()
    want = torch.empty((m, n), device=DEV, dtype=torch.bfloat16)
    _C.gemm_strided(x[:, :k].contiguous(), w[:k].t().contiguous().t(), want, config=3)
    for a in (x[:, :k], xt[:k].t()):
        got = torch.empty_like(want)
        _C.gemm_strided(a, w[:k], got, config=_lib.GEMM_CONFIGS["256x256_solo"])
        assert torch.equal(got.view(torch.int16), want.view(torch.int16))


# (tokens, inputs, outputs): one tile each, one of either and many of the other, both products longer, shares of two sizes
PAIR_SHAPES = [(8, 8, 8), (64, 264, 8200), (2304, 256, 320), (1030, 1032, 2056), (2047, 4096, 4096), (4120, 4096, 1600), (300, 16384, 4160)]


@pytest.mark.parametrize("tokens,inputs,outputs", PAIR_SHAPES)
def test_both_gradients_of_a_linear_layer(tokens, inputs, outputs):
    from rl_engine import _lib

    lib = _lib.load()
    gen = torch.Generator(device=DEV).manual_seed(tokens)
    g, x, w = (torch.randn(s, generator=gen, device=DEV, dtype=torch.bfloat16) for s in ((tokens, outputs), (tokens, inputs), (outputs, inputs)))

    def backward(config):
        dx, dw = torch.full_like(x, 7.0), torch.full_like(w, 7.0)
        stream = torch.cuda.current_stream().cuda_stream
        assert lib.rlk_linear_bwd_bf16(g.data_ptr(), outputs, x.data_ptr(), inputs, w.data_ptr(), inputs, dx.data_ptr(), inputs,
                                       dw.data_ptr(), inputs, tokens, inputs, outputs, config, stream) == 0  # fmt: skip
        return dx.view(torch.int16), dw.view(torch.int16)

    want = backward(1)
    for config in (_lib.LINEAR_BWD_SOLO, _lib.LINEAR_BWD_SOLO_192, _lib.LINEAR_BWD_SOLO_128, 0):
        got = backward(config)
        assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])


@pytest.mark.parametrize("tokens,vocab", [(2050, 12337), (4120, 9000)])
def test_gradients_of_the_logp_at_a_ragged_vocabulary(tokens, vocab):
    """Sizes where they run in one launch of these tiles: the bits of each gradient asked for alone."""
    from rl_engine import _C

    gen = torch.Generator(device=DEV).manual_seed(tokens)
    h = torch.randn((tokens, 2048), generator=gen, device=DEV, dtype=torch.bfloat16)
    w = torch.randn((vocab, 2048), generator=gen, device=DEV, dtype=torch.bfloat16).mul_(0.02)
    ids = torch.randint(0, vocab, (tokens,), generator=gen, device=DEV)
    _, lse = _C.fused_linear_logp(h, w, ids)
    grad = torch.randn(tokens, generator=gen, device=DEV)
    both = _C.fused_linear_logp_bwd(h, w, ids, lse, grad, None)
    hidden = _C.fused_linear_logp_bwd(h, w, ids, lse, grad, None, need_grad_weight=False)
    weight = _C.fused_linear_logp_bwd(h, w, ids, lse, grad, None, need_grad_hidden=False)
    assert torch.equal(both[0].view(torch.int16), hidden[0].view(torch.int16))
    assert torch.equal(both[1].view(torch.int16), weight[1].view(torch.int16))


# (tokens, vocabulary, hidden): one more token than 64, tiles of 128, 192 and 256 tokens at their edges, a vocabulary that ends inside a
# split's first slice, inside its second tile, on a tile; more tiles than compute units
STREAM_SHAPES = [(65, 1030, 64), (128, 2304, 192), (129, 2100, 128), (192, 50257, 64), (193, 9000, 256), (257, 8192, 64), (300, 18992, 128),
                 (640, 37984, 64), (1000, 20001, 128), (1024, 33000, 64)]  # fmt: skip


@pytest.mark.parametrize("shape", STREAM_SHAPES)
@pytest.mark.parametrize("temperature", [False, True])
@pytest.mark.parametrize("padded", [0, 7])  # columns of the vocabulary that are not real
def test_stream_groups_of_the_logp(shape, temperature, padded):
    """Up to 1024 tokens: the bits of the eight-wave kernel that keeps a split to one workgroup, with and without the logits."""
    from rl_engine import _C

    t, v, d = shape
    gen = torch.Generator(device=DEV).manual_seed(t + v)
    h = torch.randn((t, d), generator=gen, device=DEV, dtype=torch.bfloat16)
    w = torch.randn((v, d), generator=gen, device=DEV, dtype=torch.bfloat16).mul_(0.1)
    ids = torch.randint(0, v - padded, (t,), generator=gen, device=DEV)
    ids[:2] = torch.tensor([0, v - padded - 1], device=DEV)
    temp = torch.rand(t, generator=gen, device=DEV) + 0.5 if temperature else None
    want = _C.fused_linear_logp(h, w, ids, None, temp, True, v - padded, config=1)  # 256 tokens, a split to a workgroup
    plain = _C.fused_linear_logp(h, w, ids, None, temp, False, v - padded)
    logits = torch.empty(t, _C.linear_logp_logits_row_stride(v), device=DEV)
    kept = _C.fused_linear_logp_into(h, w, ids, None, temp, v - padded, logits)
    for got in (plain, kept):
        assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
    assert torch.equal(logits[:, :v], want[2])
