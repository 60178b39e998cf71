"""Which kernels the automatic choices launch, by the names that a trace of the call shows: the rules at the sizes where they turn."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda"


def launched(call) -> list[str]:
    """The kernels of ``call``, in order."""
    call()  # the first call's allocations and attributes are not of interest
    torch.cuda.synchronize()
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU, torch.profiler.ProfilerActivity.CUDA]) as trace:
        call()
        torch.cuda.synchronize()
    events = [e for e in trace.events() if e.device_type == torch.autograd.DeviceType.CUDA]
    names = [e.name for e in sorted(events, key=lambda e: e.time_range.start)]
    assert names, "the trace holds no kernel"
    return names


def _rand(*shape):
    return torch.randn(shape, device=DEV, dtype=torch.bfloat16)


# (tokens, vocabulary, hidden, stored logits, four waves); 76, 128, 132, 152, 260 and 512 tiles of weights below and from 192 MiB (with
# stored logits) and 224 MiB, a vocabulary of half a split and one more
@pytest.mark.parametrize(
    "tokens,vocab,hidden,logits,four",
    [(96, 18992, 64, False, True), (96, 18992, 64, True, True), (96, 32768, 64, False, True), (128, 33000, 64, True, True),
     (128, 33000, 3072, True, False), (128, 33000, 3072, False, True), (96, 37984, 3072, False, True),
     (96, 37984, 3136, False, False), (65, 66000, 1024, True, True), (65, 66000, 1600, True, False), (65, 66000, 1600, False, True),
     (96, 131072, 64, True, True), (96, 131072, 64, False, True), (100, 512, 64, False, False), (100, 500, 64, True, False),
     (100, 513, 64, True, True), (300, 512, 64, False, False), (300, 513, 64, True, True), (200, 512, 64, True, True)],
)  # fmt: skip
def test_stream_groups_of_the_logp(tokens, vocab, hidden, logits, four):
    from rl_engine import _C

    h, w = _rand(tokens, hidden), _rand(vocab, hidden)
    ids = torch.zeros(tokens, dtype=torch.int64, device=DEV)
    out = torch.empty(tokens, _C.linear_logp_logits_row_stride(vocab), device=DEV)
    if logits:
        names = launched(lambda: _C.fused_linear_logp_into(h, w, ids, None, None, vocab, out))
    else:
        names = launched(lambda: _C.fused_linear_logp(h, w, ids, None, None, False, vocab))
    assert any("linear_logp_streamgroup_solo_kernel" in n for n in names) == four
    assert any("linear_logp_streamgroup_kernel" in n for n in names) != four


# (tokens, outputs, K, operand, configuration): reductions that 64 divides and 128 does not, as small tiles; what the four-wave forms
# do not take - rows off 16 bytes, fp32 results, the staged loop - as the shapes of eight waves; a single K tile in one round
@pytest.mark.parametrize(
    "tokens,outputs,k,operand,config",
    [(65, 2880, 2880, "native", "64x64"), (300, 2880, 1600, "native", "64x64"), (441, 5000, 64, "native", "128x128"),
     (104, 1536, 1600, "pitch", "64x64"), (1452, 4096, 320, "pitch", "192x128"), (830, 4096, 64, "pitch", "128x128"), (189, 6144, 2880, "pitch", "128x64"), (241, 12288, 1600, "pitch", "128x128"),
     (65, 2880, 2880, "fp32", "64x64"), (600, 1536, 1600, "staged", "64x64"), (1822, 5760, 64, "native", "256x192"),
     (1590, 4096, 64, "native", "256x128"), (6000, 5760, 64, "native", "192x256 four"),
     (2047, 4096, 2880, "native", "192x192 four"), (1822, 5760, 128, "native", "256x192 four")],
)  # fmt: skip
def test_tiles_of_a_projection(tokens, outputs, k, operand, config):
    from rl_engine import _C, _lib

    pad = 1 if operand == "pitch" else 0
    x, w = _rand(tokens, k + pad)[:, :k], _rand(outputs, k + pad)[:, :k]
    out = torch.empty((tokens, outputs), device=DEV, dtype=torch.float32 if operand == "fp32" else torch.bfloat16)
    name, _, four = config.partition(" ")
    asked = _lib.GEMM_CONFIGS[name] | (_lib.FOUR_WAVES if four else 0)
    staged = _lib.FORCE_STAGED if operand == "staged" else 0
    auto = launched(lambda: _C.gemm_strided(x, w.t(), out, config=staged))
    assert auto == launched(lambda: _C.gemm_strided(x, w.t(), out, config=asked | staged))
    assert len(auto) == 1 and ("det_gemm_solo_kernel" in auto[0]) == bool(four)


# K-major weights (rows of a multiple of 4 KiB that is no power of two: 6144, 12288 outputs): 256 x 128 and 256 x 192 with four waves or
# with eight
@pytest.mark.parametrize(
    "tokens,outputs,config",
    [(1024, 8192, "256x128 four"), (1000, 5128, "256x128 four"), (640, 12288, "256x128"), (1100, 6144, "256x128"),
     (700, 12288, "256x192"), (1500, 6144, "256x192"), (700, 13312, "256x192 four"), (3400, 6144, "256x192 four")],
)  # fmt: skip
def test_tiles_of_a_kmajor_weight(tokens, outputs, config):
    from rl_engine import _C, _lib

    k = 256
    x, w = _rand(tokens, k), _rand(k, outputs)
    out = torch.empty((tokens, outputs), device=DEV, dtype=torch.bfloat16)
    name, _, four = config.partition(" ")
    auto = launched(lambda: _C.gemm_strided(x, w, out))
    assert auto == launched(lambda: _C.gemm_strided(x, w, out, config=_lib.GEMM_CONFIGS[name] | (_lib.FOUR_WAVES if four else 0)))
    assert len(auto) == 1 and ("det_gemm_solo_kernel" in auto[0]) == bool(four)


# what rlk_linear_bwd_pick_solo() names is what runs, four waves and eight
@pytest.mark.parametrize("tokens,inputs,outputs", [(2047, 4096, 4096), (1508, 4096, 4096), (1024, 4096, 4096), (8192, 1024, 1024), (128, 4096, 4096)])
def test_launches_of_a_linear_backward(tokens, inputs, outputs):
    from rl_engine import _lib

    lib = _lib.load()
    g, x, w = _rand(tokens, outputs), _rand(tokens, inputs), _rand(outputs, inputs)
    dx, dw = torch.empty_like(x), torch.empty_like(w)

    def backward(config):
        assert 0 == lib.rlk_linear_bwd_bf16(g.data_ptr(), outputs, x.data_ptr(), inputs, w.data_ptr(), inputs, dx.data_ptr(), inputs,
                                            dw.data_ptr(), inputs, tokens, inputs, outputs, config, torch.cuda.current_stream().cuda_stream)  # fmt: skip

    solo = lib.rlk_linear_bwd_pick_solo(tokens, inputs, outputs, 0)
    auto = launched(lambda: backward(0))
    assert auto == launched(lambda: backward(solo or lib.rlk_linear_bwd_pick_config(tokens, inputs, outputs, 0)))
    assert any("det_gemm_pair_solo_kernel" in n for n in auto) == (solo != 0)


# the kernels that the large shapes run by the automatic choices: on four waves, and on eight with few tiles
def test_kernels_of_the_large_shapes():
    from rl_engine import _C, _lib

    lib = _lib.load()

    def one(call, kernel):
        names = [n for n in launched(call) if "merge" not in n]
        assert any(kernel in n for n in names), names

    x, w = _rand(4096, 256), _rand(4096, 256)
    out = torch.empty((4096, 4096), device=DEV, dtype=torch.bfloat16)
    one(lambda: _C.gemm_strided(x, w.t(), out), "det_gemm_solo_kernel")
    one(lambda: _C.gemm_strided(x, w.t().contiguous(), out), "det_gemm_solo_kernel")
    few = torch.empty((1024, 2048), device=DEV, dtype=torch.bfloat16)  # 32 tiles
    one(lambda: _C.gemm_strided(x[:1024], w[:2048].t(), few, config=1), "det_gemm_kernel")
    one(lambda: _C.det_gemm_swiglu(x, w), "det_gemm_swiglu_solo_kernel")
    y = [torch.empty((4096, 4096), device=DEV, dtype=torch.bfloat16) for _ in range(3)]
    stream = torch.cuda.current_stream().cuda_stream
    one(lambda: lib.rlk_det_gemm_swiglu_training_bf16(x.data_ptr(), 256, w.data_ptr(), w.data_ptr(), 256, *(t.data_ptr() for t in y), 4096,
                                                      4096, 4096, 256, stream), "det_gemm_swiglu_solo_kernel")  # fmt: skip


# LogP above 1024 tokens: units on four waves, with a bias or few units on eight; both gradients in one launch of them
@pytest.mark.parametrize("tokens,vocab,bias,logits,four", [(2048, 50257, False, False, True), (4000, 18992, False, True, True),
                                                           (2048, 50257, True, False, False), (2048, 37984, False, False, False),
                                                           # a rest of up to 128 tokens: whose units open a round behind one or two, or with
                                                           # stored logits just above one round; and the nearest that don't
                                                           (2126, 32768, False, False, False), (2110, 32768, False, True, True), (2060, 32768, False, False, True),
                                                           (3430, 37984, False, True, True), (1640, 37984, False, True, True), (1640, 37984, False, False, False),
                                                           (2311, 32768, False, True, False), (2320, 37984, False, True, True)])  # fmt: skip
def test_units_of_the_logp(tokens, vocab, bias, logits, four):
    from rl_engine import _C

    h, w = _rand(tokens, 64), _rand(vocab, 64)
    ids = torch.zeros(tokens, dtype=torch.int64, device=DEV)
    b = torch.zeros(vocab, device=DEV) if bias else None
    out = torch.empty(tokens, _C.linear_logp_logits_row_stride(vocab), device=DEV)
    if logits:
        names = launched(lambda: _C.fused_linear_logp_into(h, w, ids, b, None, vocab, out))
    else:
        names = launched(lambda: _C.fused_linear_logp(h, w, ids, b, None, False, vocab))
    assert any("linear_logp_solo_kernel" in n for n in names) == four
    assert any("linear_logp_partial_kernel" in n for n in names) != four


@pytest.mark.parametrize("tokens,vocab", [(2050, 12337), (4120, 9000), (300, 9000)])
def test_launches_of_the_logp_backward(tokens, vocab):
    from rl_engine import _C, _lib

    h, w = _rand(tokens, 2048), _rand(vocab, 2048).mul_(0.02)
    ids = torch.zeros(tokens, dtype=torch.int64, device=DEV)
    _, lse = _C.fused_linear_logp(h, w, ids)
    grad = torch.ones(tokens, device=DEV)
    names = launched(lambda: _C.fused_linear_logp_bwd(h, w, ids, lse, grad, None))
    assert any("det_gemm_pair_solo_kernel" in n for n in names) == (_lib.load().rlk_linear_bwd_pick_solo(tokens, 2048, vocab, 1) != 0)
