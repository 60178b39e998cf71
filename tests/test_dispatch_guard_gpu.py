"""A guard on the automatic tile choice of rlk_det_gemm_bf16, not a benchmark: on seeded shapes outside the
Qwen3-8B projections the picker was fitted to (odd feature counts, K = 5120 / 7168 / 14336, 300 ... 9000 tokens)
the automatic configuration must be within 1.3 x of the best forced tile configuration. Every configuration
computes the same bits (checked here as well), so a bad pick is a performance bug only - and this is what keeps it
from going unnoticed."""

from __future__ import annotations

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda"
SLACK = 1.3
FORCED = ("256x256", "192x256", "256x192", "192x192", "256x128", "192x128", "256x64", "128x128", "128x64", "64x64",
          "64x64_deep", "96x64_deep", "128x64_deep", "128x128_deep")  # fmt: skip


def _median_us(fn, launches: int) -> float:
    for _ in range(2):
        fn()
    pairs = [(torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)) for _ in range(launches)]
    torch.cuda.synchronize()
    for start, stop in pairs:
        start.record()
        fn()
        stop.record()
    torch.cuda.synchronize()
    return float(np.median([start.elapsed_time(stop) for start, stop in pairs])) * 1e3


def _shapes():
    rng = np.random.default_rng(20250)
    features = [5120, 7168, 14336, 2560, 1000, 3333, 8192, 10240, 1536, 28672, 9728, 640]
    reductions = [5120, 7168, 14336, 2560, 8192, 1024]
    out = []
    for case in range(30):
        n = int(features[case % len(features)])
        k = int(reductions[int(rng.integers(0, len(reductions)))])
        m = int(rng.integers(300, 9001))
        if m * n > 120e6 or n * k > 250e6:  # keep a case at a few hundred MB
            m = max(300, int(120e6 // n))
            k = min(k, int(250e6 // n) // 64 * 64)
        out.append((m, n, k))
    return out


def test_auto_is_close_to_the_best_forced_configuration():
    from rl_engine import _C, _lib

    worst = []
    for case, (m, n, k) in enumerate(_shapes()):
        gen = torch.Generator(device=DEV).manual_seed(7000 + case)  # drawn on the device: the values do not matter here
        a = torch.randn((m, k), generator=gen, device=DEV, dtype=torch.float32).to(torch.bfloat16)
        w = (torch.randn((n, k), generator=gen, device=DEV, dtype=torch.float32) * 0.02).to(torch.bfloat16)
        out = torch.empty((m, n), dtype=torch.bfloat16, device=DEV)
        want = torch.empty_like(out)
        _C.gemm_strided(a, w.t(), want, config=0)

        def timed(code, launches=5):
            return _median_us(lambda: _C.gemm_strided(a, w.t(), out, config=code), launches)

        auto = timed(0)
        best_name, best = "auto", auto
        for name in FORCED:
            code = _lib.GEMM_CONFIGS[name]
            us = timed(code)
            assert torch.equal(out.view(torch.int16), want.view(torch.int16)), (m, n, k, name)
            if us < best:
                best_name, best = name, us
        if auto > SLACK * best:  # one more look with more launches before calling it a bad pick
            auto, best = timed(0, 15), timed(_lib.GEMM_CONFIGS[best_name], 15)
        worst.append((auto / best, m, n, k, best_name, round(auto, 1), round(best, 1)))
        del a, w, out, want
    worst.sort(reverse=True)
    print("auto / best forced, worst five:", worst[:5])
    assert worst[0][0] <= SLACK, worst[:5]


def test_the_backward_plan_is_close_to_the_best_configuration():
    """The same for rlk_linear_bwd_bf16, whose estimate was fitted to other layers: odd and large layers, 100 to 6000 tokens."""
    from rl_engine import _lib

    lib = _lib.load()
    stream = torch.cuda.current_stream().cuda_stream
    rng = np.random.default_rng(31)
    layers = [(2560, 9728), (5120, 5120), (3584, 18944), (1000, 3336), (7168, 2048), (5120, 13824), (8192, 10240), (640, 2560)]
    worst = []
    for case in range(24):
        k, n = layers[case % len(layers)]
        m = int(round(100 * 60 ** rng.random()))
        gen = torch.Generator(device=DEV).manual_seed(case)
        g, x, w = (torch.randn(s, generator=gen, device=DEV, dtype=torch.bfloat16) for s in ((m, n), (m, k), (n, k)))
        dx, dw = torch.empty_like(x), torch.empty_like(w)

        def run(config):
            status = lib.rlk_linear_bwd_bf16(
                g.data_ptr(), n, x.data_ptr(), k, w.data_ptr(), k, dx.data_ptr(), k, dw.data_ptr(), k, m, k, n, config, stream
            )
            _lib.check(status, "rlk_linear_bwd_bf16 failed")

        times = {c: _median_us(lambda: run(c), 5) for c in range(9)}
        best = min(times, key=times.get)
        if times[0] > SLACK * times[best]:
            times[0], times[best] = _median_us(lambda: run(0), 15), _median_us(lambda: run(best), 15)
        worst.append((times[0] / times[best], m, k, n, best, round(times[0], 1), round(times[best], 1)))
    worst.sort(reverse=True)
    print("auto / best configuration, worst five:", worst[:5])
    assert worst[0][0] <= SLACK, worst[:5]
