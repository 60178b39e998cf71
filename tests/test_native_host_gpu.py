"""The native host side against the general way: the same bits of results and gradients, and the general way for everything that
is more than values in memory."""

from __future__ import annotations

import threading

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda"


class _Nothing:
    def __getattr__(self, name):
        return lambda *args: None


@pytest.fixture()
def general(monkeypatch):
    """A function that runs its argument the general way."""
    from rl_engine import _host

    def run(call):
        with monkeypatch.context() as m:
            m.setattr(_host, "_native", _Nothing())
            return call()

    return run


def _bits(t):
    return t.detach().contiguous().view(torch.int16 if t.element_size() == 2 else torch.int32)


def _same(got, want):
    assert len(got) == len(want)
    for g, w in zip(got, want):
        assert (g is None) == (w is None)
        if g is not None:
            assert g.shape == w.shape and g.dtype == w.dtype and torch.equal(_bits(g), _bits(w))


def _normal(*shape, seed=0, dtype=torch.bfloat16, scale=1.0):
    gen = torch.Generator(device=DEV).manual_seed(seed)
    return torch.randn(shape, generator=gen, device=DEV, dtype=dtype).mul_(scale)


@pytest.mark.parametrize("m,k,n", [(1, 8, 8), (1, 1024, 1536), (7, 64, 100), (333, 256, 512), (2, 3, 5)])
def test_linear(general, m, k, n):
    from rl_engine import _host
    from rl_engine.ops.gemm import DetGemmOp

    x, w, gy = _normal(m, k, seed=1), _normal(n, k, seed=2, scale=0.1), _normal(m, n, seed=3)
    op = DetGemmOp()
    assert _host.native().linear(x, w) is not None
    _same([op.linear(x, w)], general(lambda: [op.linear(x, w)]))

    def train(need):
        a, b = x.clone().requires_grad_(need[0]), w.clone().requires_grad_(need[1])
        y = op.linear(a, b)
        return [y, *torch.autograd.grad(y, [t for t in (a, b) if t.requires_grad], gy)]

    for need in ((True, True), (True, False), (False, True)):
        _same(train(need), general(lambda: train(need)))


def test_linear_other_layouts_devices_and_grads(general):
    from rl_engine import _host
    from rl_engine.ops.gemm import DetGemmOp

    op, native = DetGemmOp(), _host.native()
    x, w = _normal(16, 64, seed=1), _normal(32, 64, seed=2)
    for a, b in ((x.t().contiguous().t(), w), (x, w.float()), (x.cpu(), w), (x[None], w), (x[:0], w), (x, w[:, :32])):
        assert native.linear(a, b) is None
    _same([op.linear(x.t().contiguous().t(), w)], [op.linear(x, w)])

    # an expanded (stride 0) gradient, a wider one, one of fewer tokens' worth of alignment
    def train(gy, rows):
        a, b = x[:rows].clone().requires_grad_(), w.clone().requires_grad_()
        return list(torch.autograd.grad(op.linear(a, b), (a, b), gy))

    for gy, rows in ((torch.ones((), device=DEV, dtype=torch.bfloat16).expand(16, 32), 16), (_normal(32, 16, seed=4).t(), 16), (_normal(3, 32, seed=5), 3)):
        _same(train(gy, rows), general(lambda: train(gy, rows)))


@pytest.mark.parametrize("shape", [(1, 64), (40, 64), (3, 5, 64), (64,)])
def test_ffn(general, shape):
    from rl_engine import _host
    from rl_engine.ops.ffn import qwen3_ffn, qwen3_ffn_packed_inference

    x = _normal(*shape, seed=1)
    gate, up, down = (_normal(*s, seed=i, scale=0.1) for i, s in ((2, (96, 64)), (3, (96, 64)), (4, (64, 96))))
    packed = torch.cat([gate, up])
    assert _host.native().packed_ffn(x, packed, down) is not None and _host.native().ffn(x, gate, up, down) is not None
    _same([qwen3_ffn_packed_inference(x, packed, down)], general(lambda: [qwen3_ffn_packed_inference(x, packed, down)]))
    gy = _normal(*shape, seed=5)

    def train(need, grad):
        leaves = [t.clone().requires_grad_(n) for t, n in zip((x, gate, up, down), need)]
        y = qwen3_ffn(*leaves)
        return [y, *torch.autograd.grad(y, [t for t in leaves if t.requires_grad], grad)]

    for need in ((True,) * 4, (False, True, True, True), (True, False, False, False), (False, False, False, True)):
        for grad in (gy, gy.flip(0).contiguous(), torch.ones_like(gy)[..., :1].expand_as(gy)):
            _same(train(need, grad), general(lambda: train(need, grad)))


def _grpo_inputs(rows=5, cols=37, mask=True):
    f = dict(dtype=torch.float32)
    cur = _normal(rows, cols, seed=1, **f)
    keep = _normal(rows, cols, seed=5, **f) > -0.3 if mask else None
    return cur, cur + _normal(rows, cols, seed=2, scale=0.1, **f), cur + _normal(rows, cols, seed=3, scale=0.1, **f), _normal(rows, seed=4, **f), keep


@pytest.mark.parametrize("mask", [True, False])
@pytest.mark.parametrize("shape", [(1, 1), (5, 37), (64, 300)])
def test_grpo(general, mask, shape):
    from rl_engine import _host
    from rl_engine.ops.loss import grpo_ratio_kl_loss

    cur, old, ref, adv, keep = _grpo_inputs(*shape, mask)
    assert _host.native().grpo(cur, old, ref, adv, keep, 0.2, 0.01) is not None

    def run(weights):
        c = cur.clone().requires_grad_()
        o = old.clone().requires_grad_()
        out = grpo_ratio_kl_loss(c, o, ref, adv, keep, clip_eps=0.2, beta=0.05)
        assert out.loss.requires_grad and not out.ratio.requires_grad and not out.k3.requires_grad
        total = sum(w * s for w, s in zip(weights, (out.loss, out.policy_loss, out.kl)) if w)
        return [*out, *torch.autograd.grad(total, (c, o), allow_unused=True)]

    for weights in ((1.0, 0, 0), (0, 1.0, 2.0), (0.5, 0.25, 3.0)):
        _same(run(weights), general(lambda: run(weights)))
    with torch.no_grad():
        args = (cur.clone().requires_grad_(), old, ref, adv, keep)
        _same(list(grpo_ratio_kl_loss(*args)), general(lambda: list(grpo_ratio_kl_loss(*args))))


def test_grpo_gradients_of_gradients_batches_and_hooks(general):
    from rl_engine.ops.loss import grpo_ratio_kl_loss

    cur, old, ref, adv, keep = _grpo_inputs()

    def second():
        c = cur.clone().requires_grad_()
        out = grpo_ratio_kl_loss(c, old, ref, adv, keep, beta=0.1)
        (g,) = torch.autograd.grad(out.loss, c, create_graph=True)
        return [g, *torch.autograd.grad(g.square().sum(), c)]

    def batched():
        c = cur.clone().requires_grad_()
        out = grpo_ratio_kl_loss(c, old, ref, adv, keep, beta=0.1)
        return list(torch.autograd.grad(out.loss, c, torch.arange(1.0, 4.0, device=DEV), is_grads_batched=True))

    def hooks(unpack):
        c = cur.clone().requires_grad_()
        with torch.autograd.graph.saved_tensors_hooks(lambda t: t, unpack):
            out = grpo_ratio_kl_loss(c, old, ref, adv, keep, beta=0.1)
        return list(torch.autograd.grad(out.loss, c))

    for call in (second, batched, lambda: hooks(lambda t: t.clone()), lambda: hooks(lambda t: t.t().contiguous().t() if t.dim() == 2 else t)):
        for got, want in zip(call(), general(call)):
            torch.testing.assert_close(got, want, rtol=2e-6, atol=1e-8)  # a few fp32 roundings of exp where operations replace the kernel


def test_tangents_vmap_modes_and_tracing_go_the_general_way():
    from torch.autograd import forward_ad
    from torch.utils._python_dispatch import TorchDispatchMode

    from rl_engine import _host
    from rl_engine.ops.gemm import DetGemmOp

    native, op = _host.native(), DetGemmOp()
    x, w = _normal(4, 64, seed=1), _normal(8, 64, seed=2)
    with forward_ad.dual_level():
        assert native.linear(forward_ad.make_dual(x, torch.ones_like(x)), w) is None
    seen = []

    class Mode(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(str(func))
            return func(*args, **(kwargs or {}))

    with Mode():
        assert native.linear(x, w) is None
        y = op.linear(x, w)
    assert any("rocm_det_gemm_linear_inference" in s for s in seen)
    assert torch.equal(_bits(y), _bits(op.linear(x, w)))

    def inside(a):
        assert native.linear(a, w) is None
        return a.sum()

    torch.func.vmap(inside)(x[None].repeat(2, 1, 1))

    class Sub(torch.Tensor):
        pass

    assert native.linear(x.as_subclass(Sub), w) is None
    assert native.linear(torch.nn.Parameter(x), w) is not None
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]) as prof:
        op.linear(x, w)
    assert any("rocm_det_gemm_linear_inference" in e.key for e in prof.key_averages())
    from torch.fx.experimental.proxy_tensor import make_fx

    traced = make_fx(lambda a, b: op.linear(a, b))(x, w)
    assert any("rocm_det_gemm_linear_inference" in str(n.target) for n in traced.graph.nodes)


def test_errors_of_autograd_stay():
    from rl_engine.ops.gemm import DetGemmOp

    x, w = _normal(4, 64, seed=1).requires_grad_(), _normal(8, 64, seed=2).requires_grad_()
    y = DetGemmOp().linear(x, w)
    y.sum().backward()
    with pytest.raises(RuntimeError, match="second time"):
        y.sum().backward()
    y = DetGemmOp().linear(x, w)
    with torch.no_grad():
        w.mul_(2)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        y.sum().backward()


def test_streams_and_threads():
    from rl_engine.ops.ffn import qwen3_ffn_packed_inference
    from rl_engine.ops.gemm import DetGemmOp

    op = DetGemmOp()
    x, w = _normal(64, 256, seed=1), _normal(512, 256, seed=2)
    gate_up, down = _normal(256, 256, seed=3, scale=0.1), _normal(256, 128, seed=4, scale=0.1)
    want, want_ffn = op.linear(x, w), qwen3_ffn_packed_inference(x, gate_up, down)
    torch.cuda.synchronize()
    bad = []

    def work():
        stream = torch.cuda.Stream()
        with torch.cuda.stream(stream), torch.no_grad():
            for _ in range(50):
                a, b = op.linear(x, w), qwen3_ffn_packed_inference(x, gate_up, down)
                if not (torch.equal(a, want) and torch.equal(b, want_ffn)):
                    bad.append(1)

    threads = [threading.Thread(target=work) for _ in range(4)]
    [t.start() for t in threads]
    [t.join() for t in threads]
    assert not bad


def test_captured_calls_replay():
    from rl_engine.ops.ffn import qwen3_ffn_packed_inference
    from rl_engine.ops.gemm import DetGemmOp

    op = DetGemmOp()
    x, w = _normal(4, 256, seed=1), _normal(512, 256, seed=2)
    gate_up, down = _normal(256, 256, seed=3, scale=0.1), _normal(256, 128, seed=4, scale=0.1)
    with torch.no_grad():
        call = lambda: (op.linear(x, w), qwen3_ffn_packed_inference(x, gate_up, down))  # noqa: E731
        call()
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out = call()
        for seed in (7, 8, 9):
            x.copy_(_normal(4, 256, seed=seed))
            graph.replay()
            torch.cuda.synchronize()
            _same(out, call())


def test_gradients_under_create_graph(general):
    """Of a linear layer and of the FFN: values without a graph, as in the general way; of the loss: differentiable in both."""
    from rl_engine.ops.ffn import qwen3_ffn
    from rl_engine.ops.gemm import DetGemmOp
    from rl_engine.ops.loss import grpo_ratio_kl_loss

    op = DetGemmOp()
    x, w, down = (t.requires_grad_() for t in (_normal(16, 64, seed=1), _normal(128, 64, seed=2, scale=0.1), _normal(64, 128, seed=3, scale=0.1)))
    up = _normal(128, 64, seed=4, scale=0.1).requires_grad_()
    logp = torch.randn(4, 32, device=DEV).mul_(0.1).requires_grad_()
    fixed = [torch.randn(4, 32, device=DEV).mul_(0.1), torch.randn(4, 32, device=DEV).mul_(0.1), torch.randn(4, device=DEV)]

    def gradients():
        y, f = op.linear(x, w), qwen3_ffn(x, w, up, down)
        loss = grpo_ratio_kl_loss(logp, *fixed, beta=0.1).loss
        return [
            *torch.autograd.grad(y, (x, w), torch.ones_like(y), create_graph=True),
            *torch.autograd.grad(f, (x, w, up, down), torch.ones_like(f), create_graph=True),
            *torch.autograd.grad(loss, logp, create_graph=True),
        ]

    got, want = gradients(), general(gradients)
    assert [g.requires_grad for g in got] == [g.requires_grad for g in want] == [False] * 6 + [True]
    _same(got[:6], want[:6])
    torch.testing.assert_close(got[6], want[6], rtol=0, atol=0)
