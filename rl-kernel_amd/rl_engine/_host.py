"""The native host side of the smallest calls (csrc/torch_host.cpp), bound to the loaded library on first use."""

from __future__ import annotations

import ctypes

from rl_engine import _lib

_ENTRIES = (
    "rlk_last_error", "rlk_det_gemm_bf16", "rlk_linear_bwd_bf16", "rlk_det_gemm_swiglu_workspace_bytes", "rlk_det_gemm_swiglu_bf16",
    "rlk_det_gemm_swiglu_training_bf16", "rlk_swiglu_bwd", "rlk_grpo_workspace_bytes", "rlk_grpo_ratio_kl_loss", "rlk_grpo_ratio_kl_loss_bwd",
)  # fmt: skip
_native = None


def native():
    """The module, whose functions answer ``None`` to arguments that are not everyday ones."""
    global _native
    if _native is None:
        lib = _lib.load()
        try:
            from rl_engine import _torch_host
        except ImportError as missing:
            raise _lib.RlkLibraryMissing(
                f"rl_engine/_torch_host.so could not be loaded ({missing}): build it with `python rl-kernel_amd/build.py`"
            ) from missing
        from rl_engine.backends.rocm.ffn.ffn import ffn_gradients
        from rl_engine.backends.rocm.gemm.det_gemm import linear_gradients
        from rl_engine.backends.rocm.loss.grpo import _elementwise_gradient

        addresses = {name: ctypes.cast(getattr(lib, name), ctypes.c_void_p).value for name in _ENTRIES}
        _torch_host.bind(addresses, linear_gradients, ffn_gradients, _elementwise_gradient)
        _native = _torch_host
    return _native
