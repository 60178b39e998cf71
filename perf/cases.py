"""Performance cases of the deterministic dense path: what a rollout engine or a trainer has it do.

Every case is one call (or one forward and backward) through a public entry point of ``rl_engine``. The shapes
are those of the Qwen3-8B layers, of their tensor-parallel shards, and of the other layers and vocabularies that
published results of this path are quoted on; token counts are what batching and packing leave, so they are rarely round.

Kinds:

``projection``        inference ``x @ weight.T`` (``DetGemmOp().linear``): decode steps, prefill chunks, packed batches
``projection_train``  the same under autograd: output, input gradient and weight gradient
``ffn``               packed gated FFN of a rollout engine (``qwen3_ffn_packed_inference``)
``ffn_train``         the differentiable gated FFN with the gradients of its three weights
``logp``              fused lm_head + log-softmax + gather of sampled ids: scoring of rollouts, decode log-probs
``logp_train``        the GRPO step on top of it: log-probs, ratio / k3-KL / clipped loss, gradients of hidden and lm_head
``logits``            log-probs of logits that exist already (a sampler's), with or without their gradient
``grpo``              the loss on log-probs alone: loss, ratio, k3 and the gradient of the log-probs
``tree``              the k-tree contract (results that do not depend on the tensor-parallel degree)
"""

import math
import os
import sys

import torch

_PACKAGE = os.path.join(os.getcwd(), "rl-kernel_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

from rl_engine.backends.rocm.gemm.det_gemm import tree_gemm  # noqa: E402
from rl_engine.ops.ffn import qwen3_ffn, qwen3_ffn_packed_inference  # noqa: E402
from rl_engine.ops.gemm import DetGemmOp  # noqa: E402
from rl_engine.ops.logprob import deterministic_linear_logp, deterministic_logp_from_logits  # noqa: E402
from rl_engine.ops.loss import grpo_ratio_kl_loss  # noqa: E402

_BF16 = torch.bfloat16
_DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}

# (in, out) of linear layers: qkv, o, gate_up, down of Qwen3-8B; the same under tensor parallelism; layers of the
# published tables; the small square of the repository's first configuration.
_LAYERS = [
    (4096, 6144), (4096, 4096), (4096, 24576), (12288, 4096),
    (4096, 1536), (1024, 4096), (3072, 4096), (4096, 12288), (4096, 14336), (14336, 4096), (1024, 1024),
]  # fmt: skip
# (hidden, intermediate): Qwen3-8B, its shards of 4 and 2, a smaller model
_FFNS = [(4096, 12288), (4096, 3072), (4096, 6144), (2048, 6144)]
# (vocabulary, hidden): Qwen3-8B, shards of 8 and 4, and the vocabularies of the published linear-LogP table
_HEADS = [(151936, 4096), (18992, 4096), (37984, 4096), (131072, 2048), (50257, 2048), (32768, 2048)]
_LOGITS_VOCABS = [151936, 131072, 32768, 32000]


def listed():
    return [
        # one sequence decoding: the smallest call, a weight read once for one token
        {"name": "qkv_1_token", "kind": "projection", "tokens": 1, "in": 4096, "out": 6144},
        # a chunk of a prompt next to decoding sequences
        {"name": "down_333_tokens", "kind": "projection", "tokens": 333, "in": 12288, "out": 4096},
        # a full packed batch of ragged sequences
        {"name": "qkv_16384_tokens", "kind": "projection", "tokens": 16384, "in": 4096, "out": 6144},
        # a decode step of 64 rollouts
        {"name": "ffn_64_tokens", "kind": "ffn", "tokens": 64, "hidden": 4096, "inter": 12288},
        # attention output projection in a training micro-batch of ragged sequences
        {"name": "o_proj_train_2047_tokens", "kind": "projection_train", "tokens": 2047, "in": 4096, "out": 4096},
        # the FFN of one layer in training
        {"name": "ffn_train_4096_tokens", "kind": "ffn_train", "tokens": 4096, "hidden": 4096, "inter": 12288},
        # log-probs of the ids a sampler just drew, at its temperature
        {"name": "logp_16_tokens", "kind": "logp", "tokens": 16, "vocab": 151936, "hidden": 4096, "temperature": True},
        # scoring of packed rollouts
        {"name": "logp_8192_tokens", "kind": "logp", "tokens": 8192, "vocab": 151936, "hidden": 4096, "temperature": False},
        # one GRPO micro-batch of 8 rollouts through the lm_head, both ways
        {"name": "logp_train_8x515", "kind": "logp_train", "rollouts": 8, "length": 515, "vocab": 151936, "hidden": 4096},
        # log-probs from logits the model has written already, and their gradient
        {"name": "logits_2048_rows", "kind": "logits", "rows": 2048, "vocab": 151936, "dtype": "bf16", "backward": True},
        # the loss of a whole rollout batch: many small launches in a framework that is not careful
        {"name": "grpo_64x1024", "kind": "grpo", "rollouts": 64, "length": 1024, "mask": True},
        # a prefill chunk under the contract that tensor parallelism leaves unchanged
        {"name": "k_tree_qkv_509_tokens", "kind": "tree", "tokens": 509, "in": 4096, "out": 6144},
    ]  # fmt: skip


def _log_int(rng, low, high):
    """An integer from low to high, its logarithm uniform."""
    return max(low, min(high, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng):
    kind = rng.choice(
        ["projection"] * 4 + ["ffn"] * 2 + ["logp"] * 2
        + ["projection_train", "ffn_train", "logp_train", "logits", "grpo", "tree"]
    )  # fmt: skip
    case = {"kind": kind}
    if kind in ("projection", "projection_train", "tree"):
        low, high = {"projection": (1, 16384), "projection_train": (64, 8192), "tree": (1, 1024)}[kind]
        case["tokens"] = _log_int(rng, low, high)
        case["in"], case["out"] = rng.choice(_LAYERS)
    elif kind in ("ffn", "ffn_train"):
        case["tokens"] = _log_int(rng, 1, 8192) if kind == "ffn" else _log_int(rng, 64, 4096)
        case["hidden"], case["inter"] = rng.choice(_FFNS)
    elif kind == "logp":
        case["tokens"] = _log_int(rng, 1, 8192)
        case["vocab"], case["hidden"] = rng.choice(_HEADS)
        case["temperature"] = rng.random() < 0.5
    elif kind == "logp_train":
        case["rollouts"] = rng.choice([4, 8, 16])
        case["length"] = _log_int(rng, 16, 4096 // case["rollouts"])
        case["vocab"], case["hidden"] = rng.choice(_HEADS)
    elif kind == "logits":
        case["rows"] = _log_int(rng, 1, 4096)
        case["vocab"] = rng.choice(_LOGITS_VOCABS)
        case["dtype"] = rng.choice(["bf16", "bf16", "fp16", "fp32"])
        case["backward"] = rng.random() < 0.6
    else:
        case["rollouts"] = _log_int(rng, 4, 512)
        case["length"] = _log_int(rng, 32, 2048)
        case["mask"] = rng.random() < 0.7
    return case


def _normal(gen, *shape, scale=1.0, dtype=_BF16):
    t = torch.randn(shape, generator=gen, device="cuda", dtype=dtype)
    return t if scale == 1.0 else t.mul_(scale)


def _log_probs(hidden, weight, targets):
    """Plain log-probs of the targets, to stand the old and reference log-probs near: in blocks of tokens."""
    parts = []
    for at in range(0, hidden.size(0), 1024):
        z = (hidden[at : at + 1024] @ weight.t()).float()
        parts.append(z.gather(1, targets[at : at + 1024, None])[:, 0] - z.logsumexp(1))
    return torch.cat(parts)


def _completion_mask(gen, rollouts, length):
    """Completions end somewhere in the second half of the row or fill it."""
    ends = torch.randint(length // 2, 2 * length, (rollouts, 1), generator=gen, device="cuda")
    return torch.arange(length, device="cuda")[None, :] < ends


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    kind = case["kind"]
    state = {"kind": kind}
    if kind in ("projection", "projection_train", "tree"):
        state["x"] = _normal(gen, case["tokens"], case["in"])
        state["w"] = _normal(gen, case["out"], case["in"], scale=0.02)
        if kind != "tree":
            state["op"] = DetGemmOp()
        if kind == "projection_train":
            state["gy"] = _normal(gen, case["tokens"], case["out"], scale=0.02)
            state["x"].requires_grad_()
            state["w"].requires_grad_()
    elif kind == "ffn":
        state["x"] = _normal(gen, case["tokens"], case["hidden"])
        state["gate_up"] = _normal(gen, 2 * case["inter"], case["hidden"], scale=0.02)
        state["down"] = _normal(gen, case["hidden"], case["inter"], scale=0.02)
    elif kind == "ffn_train":
        state["x"] = _normal(gen, case["tokens"], case["hidden"]).requires_grad_()
        state["gate"] = _normal(gen, case["inter"], case["hidden"], scale=0.02).requires_grad_()
        state["up"] = _normal(gen, case["inter"], case["hidden"], scale=0.02).requires_grad_()
        state["down"] = _normal(gen, case["hidden"], case["inter"], scale=0.02).requires_grad_()
        state["gy"] = _normal(gen, case["tokens"], case["hidden"], scale=0.02)
    elif kind in ("logp", "logp_train"):
        tokens = case["tokens"] if kind == "logp" else case["rollouts"] * case["length"]
        state["hidden"] = _normal(gen, tokens, case["hidden"])
        state["head"] = _normal(gen, case["vocab"], case["hidden"], scale=0.02)
        state["ids"] = torch.randint(0, case["vocab"], (tokens,), generator=gen, device="cuda")
        state["temperature"] = None
        if case.get("temperature"):
            state["temperature"] = torch.empty(tokens, device="cuda").uniform_(0.6, 1.2, generator=gen)
        if kind == "logp_train":
            rows = (case["rollouts"], case["length"])
            near = _log_probs(state["hidden"], state["head"], state["ids"]).view(rows)
            state["old"] = near + _normal(gen, *rows, scale=0.05, dtype=torch.float32)
            state["ref"] = near + _normal(gen, *rows, scale=0.05, dtype=torch.float32)
            state["advantages"] = _normal(gen, case["rollouts"], dtype=torch.float32)
            state["mask"] = _completion_mask(gen, *rows)
            state["hidden"].requires_grad_()
            state["head"].requires_grad_()
    elif kind == "logits":
        dtype = _DTYPES[case["dtype"]]
        state["logits"] = _normal(gen, case["rows"], case["vocab"], scale=1.3, dtype=dtype)
        state["ids"] = torch.randint(0, case["vocab"], (case["rows"],), generator=gen, device="cuda")
        state["grad"] = None
        if case["backward"]:
            state["logits"].requires_grad_()
            state["grad"] = _normal(gen, case["rows"], scale=1e-3, dtype=torch.float32)
    else:
        rows = (case["rollouts"], case["length"])
        current = -torch.empty(rows, device="cuda").exponential_(0.7, generator=gen)
        state["old"] = current + _normal(gen, *rows, scale=0.05, dtype=torch.float32)
        state["ref"] = current + _normal(gen, *rows, scale=0.05, dtype=torch.float32)
        state["current"] = current.requires_grad_()
        state["advantages"] = _normal(gen, case["rollouts"], dtype=torch.float32)
        state["mask"] = _completion_mask(gen, *rows) if case["mask"] else None
    return state


def run(state):
    kind = state["kind"]
    if kind == "projection":
        with torch.no_grad():
            return state["op"].linear(state["x"], state["w"])
    if kind == "projection_train":
        y = state["op"].linear(state["x"], state["w"])
        dx, dw = torch.autograd.grad(y, (state["x"], state["w"]), state["gy"])
        return {"y": y, "dx": dx, "dw": dw}
    if kind == "tree":
        return tree_gemm(state["x"], state["w"].t())
    if kind == "ffn":
        with torch.no_grad():
            return qwen3_ffn_packed_inference(state["x"], state["gate_up"], state["down"])
    if kind == "ffn_train":
        y = qwen3_ffn(state["x"], state["gate"], state["up"], state["down"])
        grads = torch.autograd.grad(y, (state["x"], state["gate"], state["up"], state["down"]), state["gy"])
        return {"y": y, "dx": grads[0], "dgate": grads[1], "dup": grads[2], "ddown": grads[3]}
    if kind == "logp":
        with torch.no_grad():
            logp, lse = deterministic_linear_logp(
                state["hidden"], state["head"], state["ids"], temperature=state["temperature"]
            )
        return {"logp": logp, "lse": lse}
    if kind == "logp_train":
        logp, _ = deterministic_linear_logp(state["hidden"], state["head"], state["ids"])
        out = grpo_ratio_kl_loss(
            logp.view(state["old"].shape), state["old"], state["ref"], state["advantages"], state["mask"],
            clip_eps=0.2, beta=0.01,
        )  # fmt: skip
        dh, dw = torch.autograd.grad(out.loss, (state["hidden"], state["head"]))
        return {"logp": logp, "loss": out.loss, "kl": out.kl, "dhidden": dh, "dhead": dw}
    if kind == "logits":
        if state["grad"] is None:
            with torch.no_grad():
                logp, lse = deterministic_logp_from_logits(state["logits"], state["ids"])
            return {"logp": logp, "lse": lse}
        logp, lse = deterministic_logp_from_logits(state["logits"], state["ids"])
        (dlogits,) = torch.autograd.grad(logp, state["logits"], state["grad"])
        return {"logp": logp, "lse": lse, "dlogits": dlogits}
    out = grpo_ratio_kl_loss(
        state["current"], state["old"], state["ref"], state["advantages"], state["mask"], clip_eps=0.2, beta=0.01
    )
    (grad,) = torch.autograd.grad(out.loss, state["current"])
    return {"loss": out.loss, "policy": out.policy_loss, "kl": out.kl, "ratio": out.ratio, "k3": out.k3, "grad": grad}


def work(case):
    kind = case["kind"]
    if kind in ("projection", "tree", "projection_train"):
        m, k, n = case["tokens"], case["in"], case["out"]
        once = 2.0 * (m * k + n * k + m * n)
        if kind == "projection_train":  # x, w, dy in; y, dx, dw out
            return {"bytes": 2 * once, "flops": 6.0 * m * n * k}
        return {"bytes": once, "flops": 2.0 * m * n * k}
    if kind in ("ffn", "ffn_train"):
        t, h, i = case["tokens"], case["hidden"], case["inter"]
        if kind == "ffn":
            return {"bytes": 2.0 * (2 * t * h + 3 * h * i), "flops": 6.0 * t * h * i}
        # x, dy and three weights in; y, dx and three gradients out
        return {"bytes": 2.0 * (4 * t * h + 6 * h * i), "flops": 18.0 * t * h * i}
    if kind == "logp":
        t, v, d = case["tokens"], case["vocab"], case["hidden"]
        return {"bytes": 2.0 * (t * d + v * d) + 16.0 * t, "flops": 2.0 * t * v * d}
    if kind == "logp_train":
        t, v, d = case["rollouts"] * case["length"], case["vocab"], case["hidden"]
        return {"bytes": 4.0 * (t * d + v * d) + 21.0 * t, "flops": 6.0 * t * v * d}
    if kind == "logits":
        elements = float(case["rows"]) * case["vocab"]
        size = 4 if case["dtype"] == "fp32" else 2
        return {"bytes": elements * size * (2 if case["backward"] else 1), "flops": elements * (8 if case["backward"] else 4)}
    tokens = float(case["rollouts"]) * case["length"]
    return {"bytes": tokens * (25 if case["mask"] else 24), "flops": tokens * 20}


def tolerance(case):
    kind = case["kind"]
    if kind == "tree":
        return "exact"  # the contract fixes every rounding
    if kind == "logits" and (case["dtype"] == "fp32" or not case["backward"]):
        return {"rel": 4e-7}  # fp32 results: at most 8e-8 from the same path in 64 bits
    # about four times the largest distance of an output from the same path in 64 bits
    return {"rel": {
        "projection": 7e-3,  # 1.7e-3: the rounding to bf16
        "projection_train": 7e-3,  # 1.7e-3, every output
        "ffn": 1.5e-2,  # 3.5e-3: the projection, the activation and the output are rounded
        "ffn_train": 1.6e-2,  # 3.9e-3 (dx, a bf16 sum of two rounded products)
        "logp": 4e-7,  # 8e-8
        "logp_train": 1e-2,  # 2.3e-3 (gradients; log-probs and loss are below 3e-6)
        "logits": 9e-3,  # 2.2e-3 (fp16 gradient, partly denormal), 1.8e-3 (bf16)
        "grpo": 8e-5,  # 2.0e-5 (k3, a difference of nearly equal numbers)
    }[kind]}  # fmt: skip
