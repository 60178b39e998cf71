"""Host-side checks that need no GPU: the C ABI exports what include/rlk.h
declares, shape heuristics are pure functions, and the Python layer raises the
reference's errors before any kernel is launched."""

from __future__ import annotations

import ctypes
import re
import subprocess
import sys
from pathlib import Path

import numpy as np
import pytest
import torch

REPO_ROOT = Path(__file__).resolve().parent.parent
HEADER = REPO_ROOT / "include" / "rlk.h"


def _declared_functions() -> list[str]:
    text = re.sub(r"/\*.*?\*/", "", HEADER.read_text(), flags=re.S)
    return sorted(set(re.findall(r"\b(rlk_[a-z0-9_]+)\s*\(", text)))


def test_header_declares_the_expected_entry_points():
    names = _declared_functions()
    for required in ("rlk_det_gemm_bf16", "rlk_linear_logp_fwd", "rlk_linear_logp_fwd_shard", "rlk_grpo_ratio_kl_loss", "rlk_contract_id"):
        assert required in names


def test_library_exports_every_declared_symbol(rlk_lib):
    for name in _declared_functions():
        assert hasattr(rlk_lib, name), f"{name} declared in include/rlk.h but not exported"


def test_python_binding_lists_the_same_symbols():
    from rl_engine import _lib

    assert sorted(_lib.EXPORTED_SYMBOLS) == _declared_functions()


def test_header_compiles_as_plain_c(tmp_path):
    src = tmp_path / "use_rlk.c"
    src.write_text('#include "rlk.h"\nint main(void) { return (int)RLK_GEMM_CFG_COUNT - 14; }\n')
    subprocess.run(["gcc", "-std=c99", "-Wall", "-Werror", "-I", str(HEADER.parent), "-c", str(src), "-o", str(tmp_path / "o.o")], check=True)


def test_contract_ids_and_version(rlk_lib):
    assert rlk_lib.rlk_contract_id().decode().startswith("rlkernel.det_gemm.")
    assert rlk_lib.rlk_linear_logp_contract_id().decode().startswith("rlkernel.linear_logp.")
    assert re.fullmatch(r"\d+\.\d+\.\d+", rlk_lib.rlk_version().decode())


def test_split_count_is_a_function_of_vocab_only(rlk_lib):
    assert rlk_lib.rlk_linear_logp_split_count(151936) == 149  # ceil(151936 / 1024)
    assert rlk_lib.rlk_linear_logp_split_count(1024) == 1
    assert rlk_lib.rlk_linear_logp_split_count(1025) == 2
    assert rlk_lib.rlk_linear_logp_split_count(0) == 0
    assert rlk_lib.rlk_linear_logp_workspace_bytes(8192, 151936) == 3 * 149 * 8192 * 4
    assert rlk_lib.rlk_grpo_workspace_bytes(64) == 3 * 64 * 4


def test_config_pick_is_deterministic_and_in_range(rlk_lib):
    from rl_engine import _lib

    for m, n, k in ((1, 4096, 12288), (16, 24576, 4096), (256, 24576, 4096), (4096, 24576, 4096), (16384, 6144, 4096)):
        first = rlk_lib.rlk_det_gemm_pick_config(m, n, k)
        assert first == rlk_lib.rlk_det_gemm_pick_config(m, n, k)
        assert 1 <= first < len(_lib.GEMM_CONFIGS)
    assert rlk_lib.rlk_det_gemm_pick_config(4096, 24576, 4096) == _lib.GEMM_CONFIGS["256x256"]


# where 96 x 64 gives every one of 256 CUs at most one tile, from 17 to 256 tokens, and just beyond; all of them with a whole
# number of stages
@pytest.mark.parametrize(
    "m,n,k,name",
    [(64, 24576, 4096, "96x64_deep"), (65, 24576, 4096, "128x128_deep"), (80, 12288, 4096, "64x96_deep"), (97, 12288, 4096, "96x64_deep"),
     (120, 12288, 4096, "96x64_deep"), (128, 12288, 1152, "96x64_deep"), (120, 12289, 4096, "128x64_deep"),
     (120, 14336, 4096, "128x64_deep"), (160, 6144, 4096, "96x64_deep"), (256, 6144, 4096, "96x64_deep")],
)  # fmt: skip
def test_the_pick_names_the_few_token_tile_that_runs(rlk_lib, m, n, k, name):
    from rl_engine import _lib

    assert rlk_lib.rlk_det_gemm_pick_config(m, n, k) == _lib.GEMM_CONFIGS[name]


# A reduction that 64 divides and 128 does not has no deep tiles: small tiles where larger ones would leave most CUs without one, the
# shapes with four waves where they fill the chip
@pytest.mark.parametrize(
    "m,n,k,name",
    [(65, 2880, 2880, "64x64"), (65, 1536, 2880, "64x64"), (65, 5760, 2880, "64x64"), (100, 640, 1600, "64x64"), (300, 2880, 2880, "64x64"),
     (47, 14400, 64, "64x64"), (129, 5760, 2880, "128x64"), (600, 2880, 2880, "128x64"), (441, 5000, 64, "128x128"),
     (2047, 4096, 2880, "192x192"), (3000, 2880, 2880, "192x192"), (8192, 8192, 2880, "256x256"), (1009, 8192, 12288, "256x128")],
)  # fmt: skip
def test_the_pick_of_reductions_without_deep_tiles(rlk_lib, m, n, k, name):
    from rl_engine import _lib

    assert rlk_lib.rlk_det_gemm_pick_config(m, n, k) == _lib.GEMM_CONFIGS[name]


# (tokens, hidden size, vocabulary): two launches where they are faster (whole token tiles and whole K tiles of a weight from
# HBM), one launch in the tiles that are the faster ones, the rest behind whole tiles beside the weight gradient
@pytest.mark.parametrize(
    "t,d,v,config",
    [(512, 4096, 37984, 1), (512, 4096, 151936, 1), (304, 5120, 32000, 1), (384, 5120, 32000, 1), (1024, 2048, 131072, 1),
     (400, 4096, 18992, 6), (512, 4096, 18992, 6), (520, 4096, 37984, 6), (768, 4096, 37984, 6), (768, 4096, 151936, 6),
     (600, 5120, 32000, 6), (960, 4096, 37984, 3), (1040, 4096, 18992, 3), (2112, 4096, 37984, 2), (4120, 4096, 151936, 0x103)],
)  # fmt: skip
def test_the_launches_of_the_logp_backward(rlk_lib, t, d, v, config):
    assert rlk_lib.rlk_linear_bwd_pick_config(t, d, v, 1) == config


# (whose backward, tokens, inputs, outputs): a layer of 96 MiB right behind its forward (0) and one of an FFN's three weights (2)
# read their weight from HBM up to 272 tokens, a layer of 48 MiB right behind its forward does not
@pytest.mark.parametrize(
    "of,m,k,n,config",
    [(0, 100, 4096, 12288, 7), (0, 128, 4096, 12288, 1), (0, 193, 4096, 12288, 7), (0, 225, 4096, 12288, 7),
     (0, 256, 4096, 12288, 1), (0, 257, 4096, 12288, 1), (0, 273, 4096, 12288, 6), (0, 400, 4096, 12288, 6), (0, 193, 4096, 6144, 6),
     (2, 128, 4096, 12288, 7), (2, 193, 4096, 12288, 7), (2, 256, 4096, 12288, 7), (2, 272, 4096, 12288, 1),
     (2, 193, 4096, 6144, 7), (2, 256, 4096, 6144, 7), (2, 300, 4096, 6144, 6), (2, 193, 12288, 4096, 3)],
)  # fmt: skip
def test_the_launches_of_a_linear_backward(rlk_lib, of, m, k, n, config):
    assert rlk_lib.rlk_linear_bwd_pick_config(m, k, n, of) == config


# (whose backward, tokens, inputs, outputs): the four-wave launch, its tiles of dX in 256, 192 and 128 tokens, or none
@pytest.mark.parametrize(
    "of,m,k,n,config",
    [(0, 2047, 4096, 4096, 0x800), (0, 1508, 4096, 4096, 0x801), (0, 1024, 4096, 4096, 0x802), (0, 8192, 1024, 1024, 0),
     (0, 603, 3072, 4096, 0), (0, 128, 4096, 4096, 0), (0, 2910, 4096, 12288, 0x800), (1, 4120, 4096, 151936, 0x800),
     (1, 353, 4096, 151936, 0), (2, 4096, 4096, 12288, 0x800), (2, 300, 4096, 6144, 0),
     (0, 157, 12288, 4096, 0), (0, 256, 14336, 4096, 0), (0, 257, 14336, 4096, 0x801), (2, 129, 12288, 4096, 0), (2, 264, 12288, 4096, 0),
     (2, 448, 6144, 4096, 0), (2, 449, 6144, 4096, 0x802), (0, 1614, 2048, 2048, 0), (0, 3358, 1024, 4096, 0), (0, 2960, 4096, 1024, 0)],
)  # fmt: skip
def test_the_four_wave_launch_of_a_linear_backward(rlk_lib, of, m, k, n, config):
    assert rlk_lib.rlk_linear_bwd_pick_solo(m, k, n, of) == config


def test_unknown_backwards_have_no_choice(rlk_lib):
    assert rlk_lib.rlk_linear_bwd_pick_solo(64, 64, 64, 3) < 0 and rlk_lib.rlk_linear_bwd_pick_solo(0, 64, 64, 0) < 0
    assert rlk_lib.rlk_linear_bwd_pick_config(64, 64, 64, -1) < 0 and rlk_lib.rlk_linear_bwd_pick_config(64, 64, 64, 3) < 0


def test_argument_errors_are_reported_without_touching_the_gpu(rlk_lib):
    # Invalid arguments are rejected before any HIP call, so this runs on a CPU-only host.
    rc = rlk_lib.rlk_det_gemm_bf16(None, 4, 1, None, 1, 4, None, 4, -1, 4, 4, 0, 0, None)
    assert rc == -1 and b"negative size" in rlk_lib.rlk_last_error()
    rc = rlk_lib.rlk_det_gemm_bf16(None, -4, 1, None, 1, 4, None, 4, 2, 4, 4, 0, 0, None)
    assert rc == -1 and b"negative strides" in rlk_lib.rlk_last_error()
    rc = rlk_lib.rlk_det_gemm_bf16(None, 4, 1, None, 1, 4, None, 4, 2, 4, 4, 0, 99, None)
    assert rc == -1 and b"unknown config" in rlk_lib.rlk_last_error()
    assert rlk_lib.rlk_det_gemm_bf16(None, 4, 1, None, 1, 4, None, 4, 0, 4, 4, 0, 0, None) == 0  # empty M: no-op
    rc = rlk_lib.rlk_linear_logp_fwd(None, 8, None, 8, None, None, None, None, None, None, 0, 4, 8, 16, 0, 17, 0, None)
    assert rc == -1 and b"real_vocab_end" in rlk_lib.rlk_last_error()
    rc = rlk_lib.rlk_linear_logp_fwd(None, 8, None, 8, None, None, None, None, None, None, 0, 4, 8, 16, 0, 16, 0, None)
    assert rc == -1 and b"null hidden" in rlk_lib.rlk_last_error()
    rc = rlk_lib.rlk_grpo_ratio_kl_loss(None, None, None, None, None, 2, 4, 0.2, 0.0, None, None, None, None, 0, None)
    assert rc == -1 and b"out3" in rlk_lib.rlk_last_error()
    rc = rlk_lib.rlk_det_gemm_tree_bf16(None, 4, 1, None, 1, 4, None, 4, 2, 4, -4, None)
    assert rc == -1 and b"negative size" in rlk_lib.rlk_last_error()
    rc = rlk_lib.rlk_det_gemm_tree_bf16(None, 4, 1, None, 1, 4, None, 2, 2, 4, 4, None)
    assert rc == -1 and b"ldc >= N" in rlk_lib.rlk_last_error()
    assert rlk_lib.rlk_det_gemm_tree_bf16(None, 4, 1, None, 1, 4, None, 4, 2, 0, 4, None) == 0  # empty N: no-op
    rc = rlk_lib.rlk_swiglu_fwd(None, 8, None, 8, None, 8, 2, 8, 7, None)
    assert rc == -1 and b"unknown dtype" in rlk_lib.rlk_last_error()
    rc = rlk_lib.rlk_swiglu_bwd(None, 8, None, 8, None, 8, None, 8, None, 8, 2, 8, 0, None)
    assert rc == -1 and b"null operand" in rlk_lib.rlk_last_error()


def test_missing_library_fails_loudly(tmp_path):
    code = (
        "import os, sys\n"
        f"sys.path.insert(0, {str(REPO_ROOT / 'rl-kernel_amd')!r})\n"
        f"os.environ['RLK_LIBRARY'] = {str(tmp_path / 'nope.so')!r}\n"
        "from rl_engine import _lib\n"
        "try:\n"
        "    _lib.load()\n"
        "except _lib.RlkLibraryMissing as e:\n"
        "    assert 'no fallback' in str(e).lower()\n"
        "    sys.exit(0)\n"
        "sys.exit(1)\n"
    )
    assert subprocess.run([sys.executable, "-c", code]).returncode == 0


def test_product_never_imports_the_oracle():
    pkg = REPO_ROOT / "rl-kernel_amd"
    for path in list(pkg.rglob("*.py")) + list(pkg.rglob("*.hip")) + list(pkg.rglob("*.h")):
        text = path.read_text()
        assert "oracle" not in text.lower(), f"{path} mentions the oracle"


# ---------------------------------------------------------------------------
# Python surface: names and pre-launch validation (CPU tensors)
# ---------------------------------------------------------------------------


def test_ops_gemm_exports_the_reference_names():
    import rl_engine.ops.gemm as pkg
    import rl_engine.ops.gemm.det_gemm as mod

    assert sorted(mod.__all__) == sorted(
        [
            "DetGemmOp",
            "det_gemm_backend",
            "det_gemm_backend_id",
            "det_gemm_fallback_reason",
            "det_gemm_linear",
            "det_gemm_linear_input_gradient",
            "det_gemm_linear_weight_gradient",
            "deterministic_gemm",
        ]
    )
    assert pkg.__all__ == ["DetGemmOp", "deterministic_gemm"]
    assert mod.det_gemm_fallback_reason() is None
    assert mod.det_gemm_backend() == "hip_mfma"
    assert mod.det_gemm_backend_id().startswith("rlkernel.det_gemm.")
    from rl_engine.backends.rocm.gemm import det_gemm as facade

    for name in ("prepare_det_gemm_linear_weight", "det_gemm_linear_prepared", "refresh_cached_weight_transposes", "RocmDetGemmOp"):
        assert hasattr(facade, name)


def test_native_module_has_the_reference_function_names():
    from rl_engine import _C

    names = (
        "det_gemm_sm90_compiled", "det_gemm_fwd", "det_gemm_fwd_rhs_transposed", "det_gemm_da", "det_gemm_db",
        "det_gemm_db_transposed", "fused_linear_logp", "fused_linear_logp_sm90", "fused_linear_logp_sm90_global_target",
        "fused_linear_logp_sm90_backward", "hip_deterministic_logp_tile_stats", "hip_deterministic_logp_backward",
        "swiglu_forward", "swiglu_backward", "swiglu_packed_forward", "swiglu_packed_backward",
    )  # fmt: skip
    for name in names:
        assert callable(getattr(_C, name))
    assert _C.det_gemm_sm90_compiled() is False


def test_native_checks_use_the_reference_error_strings():
    from rl_engine import _C

    a = torch.zeros((2, 4), dtype=torch.bfloat16)
    with pytest.raises(RuntimeError, match="A must be CUDA"):
        _C.det_gemm_fwd(a, a)
    with pytest.raises(RuntimeError, match="dC must be CUDA"):
        _C.det_gemm_da(a, a)


def test_facade_validation_matches_the_reference_error_types():
    from rl_engine.backends.rocm.gemm import det_gemm as facade

    a = torch.zeros((2, 4), dtype=torch.bfloat16)
    with pytest.raises(ValueError, match="two 2-D tensors"):
        facade.mfma_gemm(a[0], a)
    with pytest.raises(ValueError, match="K mismatch"):
        facade.mfma_gemm(a, a)
    with pytest.raises(TypeError, match="requires BF16 inputs"):
        facade.mfma_gemm(a.float(), a.float().t())
    with pytest.raises(RuntimeError, match="share one ROCm device"):
        facade.mfma_gemm(a, a.t())
    op = facade.DetGemmOp()
    with pytest.raises(AssertionError, match="BF16 only"):
        op(a.float(), a.float().t())
    with pytest.raises(AssertionError, match="ROCm device"):
        op(a, a.t())
    with pytest.raises(TypeError, match="must be BF16"):
        facade.prepare_det_gemm_linear_weight(a.float())
    with pytest.raises(ValueError, match="must be 2-D"):
        facade.prepare_det_gemm_linear_weight(a[0])


def test_prepared_weight_registry_identifies_sources_by_storage():
    import gc

    from rl_engine.backends.rocm.gemm import det_gemm as facade

    w = torch.zeros((6, 4), dtype=torch.bfloat16)
    buf_a, buf_b = torch.zeros((4, 6), dtype=torch.bfloat16), torch.zeros((4, 6), dtype=torch.bfloat16)
    facade._remember_prepared(w, buf_a)
    facade._remember_prepared(w.data, buf_b)  # another tensor object over the same storage: the same source
    facade._remember_prepared(w, buf_a)  # registered once
    live = facade._live_prepared(w)
    assert len(live) == 2 and live[0] is buf_a and live[1] is buf_b
    assert facade._live_prepared(w[:3]) == [] and facade._live_prepared(w.view(4, 6)) == []  # other views: other sources
    del buf_b, live
    gc.collect()
    assert [b is buf_a for b in facade._live_prepared(w)] == [True]  # a dropped buffer is forgotten
    entries = len(facade._PREPARED_TRANSPOSES)
    del w
    gc.collect()
    assert len(facade._PREPARED_TRANSPOSES) == entries - 1  # the entry dies with the source's storage
    w2 = torch.zeros((6, 4), dtype=torch.bfloat16)  # likely the same address; a different source all the same
    assert facade._live_prepared(w2) == []


def test_linear_logp_python_validation():
    from rl_engine.ops.logprob import LinearLogpOp, deterministic_linear_logp

    h = torch.zeros((3, 8), dtype=torch.bfloat16)
    w = torch.zeros((16, 8), dtype=torch.bfloat16)
    t = torch.zeros((3,), dtype=torch.long)
    with pytest.raises(RuntimeError, match="requires a GPU tensor"):
        deterministic_linear_logp(h, w, t)
    op = LinearLogpOp()
    with pytest.raises(ValueError, match="leading shape"):
        op(h, w, t[:2])
    with pytest.raises(ValueError, match="must match lm_head_weight dim"):
        op(h, torch.zeros((16, 4), dtype=torch.bfloat16), t)


def test_ctypes_prototypes_cover_every_argument(rlk_lib):
    # A prototype with the wrong arity would corrupt the call; compare with the header.
    text = re.sub(r"/\*.*?\*/", "", HEADER.read_text(), flags=re.S)
    from rl_engine import _lib

    for name in _lib.EXPORTED_SYMBOLS:
        params = re.search(r"\b" + name + r"\s*\((.*?)\)\s*;", text, flags=re.S).group(1).strip()
        declared = 0 if params == "void" else params.count(",") + 1
        assert len(getattr(rlk_lib, name).argtypes) == declared, name
    assert rlk_lib.rlk_linear_logp_workspace_bytes.restype is ctypes.c_size_t


def test_linear_logp_wrapper_contract_errors_without_a_gpu():
    """Shape / dtype / placement rules of the engine-facing wrapper are checked before any GPU work."""
    import torch

    from rl_engine.integrations.common.linear_logp import LinearLogpWrapper

    wrapper = LinearLogpWrapper()
    ids = torch.zeros(2, dtype=torch.long)
    with pytest.raises(ValueError, match=r"expects hidden \[tokens, hidden\]"):
        wrapper(torch.zeros(3), torch.zeros(2, 3), ids)
    with pytest.raises(RuntimeError, match="requires CUDA/ROCm GPU tensors"):
        wrapper(torch.zeros(2, 3, dtype=torch.bfloat16), torch.zeros(4, 3, dtype=torch.bfloat16), ids)
    with pytest.raises(TypeError, match="2-D bf16/fp16/fp32"):
        wrapper.from_local_logits(torch.zeros(2, 8, dtype=torch.float64), ids, tp_group=None, vocab_start_index=0, global_vocab_size=8, real_vocab_size=8)
    with pytest.raises(ValueError, match="temperature must be positive"):
        LinearLogpWrapper._temperature_tensor(0.0, rows=2, device=torch.device("cpu"))
    assert LinearLogpWrapper._temperature_tensor(1.0, rows=2, device=torch.device("cpu")) is None
    with pytest.raises(ValueError, match=r"target_ids must be in \[0, 4\)"):
        LinearLogpWrapper._validate_targets(torch.tensor([0, 4]), rows=2, real_vocab_size=4)
    with pytest.raises(TypeError, match="integer dtype"):
        LinearLogpWrapper._validate_targets(torch.tensor([0.0, 1.0]), rows=2, real_vocab_size=4)
    assert wrapper.provenance == {}


def test_group_advantages_known_answers_and_errors():
    """Host-side reward normalisation: the reference's own known answer and argument checks
    (tests/ops/loss/test_grpo_loss.py:94-128), and equality with the oracle."""
    from oracle import reference_math as oracle
    from rl_engine.ops.loss import group_advantages

    got = group_advantages(torch.tensor([1.0, 3.0, 10.0, 20.0, 30.0]), group_boundaries=[0, 2, 5])
    g1 = (torch.tensor([10.0, 20.0, 30.0]) - 20.0) / (200.0 / 3.0) ** 0.5
    assert torch.allclose(got, torch.cat([torch.tensor([-1.0, 1.0]), g1]), atol=1e-5)
    rewards = torch.randn(12, generator=torch.Generator().manual_seed(61))
    uniform = group_advantages(rewards.view(3, 4), samples_per_prompt=4)
    assert uniform.shape == (12,) and uniform.dtype == torch.float32
    assert torch.allclose(uniform, group_advantages(rewards, group_boundaries=[0, 4, 8, 12]), atol=1e-6)
    assert torch.allclose(uniform, torch.from_numpy(oracle.group_advantages(rewards.numpy(), samples_per_prompt=4)), atol=1e-6)
    ragged = group_advantages(rewards, group_boundaries=torch.tensor([0, 1, 5, 12]))
    assert torch.allclose(ragged, torch.from_numpy(oracle.group_advantages(rewards.numpy(), group_boundaries=[0, 1, 5, 12])), atol=1e-5)
    # boundaries that do not start at zero: only the group sizes count (the reference builds its group ids with
    # repeat_interleave over the differences), and every sequence gets a value
    six = rewards[:6]
    shifted = group_advantages(six, group_boundaries=[2, 5, 8])
    assert torch.equal(shifted, group_advantages(six, group_boundaries=[0, 3, 6]))
    g0 = six[:3]
    want0 = (g0 - g0.mean()) / ((g0 * g0).mean() - g0.mean() ** 2).clamp_min(1e-12).sqrt()
    assert torch.allclose(shifted[:3], want0, atol=1e-5) and bool(torch.isfinite(shifted).all())
    assert np.allclose(oracle.group_advantages(six.numpy(), group_boundaries=[2, 5, 8]), shifted.numpy(), atol=1e-5)
    assert float(ragged[0]) == 0.0  # a group of one: zero variance is floored at eps, the numerator is zero
    assert torch.equal(group_advantages(torch.full((4,), 2.5), samples_per_prompt=2), torch.zeros(4))
    for kwargs in ({}, {"samples_per_prompt": 4, "group_boundaries": [0, 4, 8, 12]}, {"samples_per_prompt": 1},
                   {"samples_per_prompt": 5}, {"group_boundaries": [0, 4, 8]}, {"group_boundaries": [0, 4, 4, 12]},
                   {"group_boundaries": [12]}):  # fmt: skip
        with pytest.raises(ValueError):
            group_advantages(rewards, **kwargs)
