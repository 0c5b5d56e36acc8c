"""``hip_kernel.eager.apply`` against ``Function.apply``: the same outputs, gradients, node and refusals, by a function that keeps its
context apart."""

import pytest
import torch

from spikingjelly_amd.activation_based.hip_kernel import eager


class _Scaled(torch.autograd.Function):
    @staticmethod
    def forward(x, k, spec):
        return x * k, x.sum(0), x > 0

    @staticmethod
    def setup_context(ctx, inputs, output):
        x, k, ctx.spec = inputs
        ctx.save_for_backward(x, k, output[2])
        ctx.mark_non_differentiable(output[2])
        ctx.set_materialize_grads(False)

    @staticmethod
    def backward(ctx, grad, grad_sum, _):
        x, k, positive = ctx.saved_tensors
        assert positive.dtype == torch.bool and grad_sum is None
        return (grad * k * ctx.spec[0]) if ctx.needs_input_grad[0] else None, (grad * x).sum() if ctx.needs_input_grad[1] else None, None


def _results(apply, x_grad, k_grad, hooks):
    x = torch.arange(-3.0, 5.0).requires_grad_(x_grad)
    k = torch.tensor(1.5).requires_grad_(k_grad)
    seen = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: seen.append(tuple(t.shape)) or t.clone(), lambda t: t) if hooks else torch.enable_grad():
        out = apply(x, k, (2.0,))
    node = out[0].grad_fn.name() if out[0].requires_grad else None
    if out[0].requires_grad:
        out[0].square().sum().backward()
    return [o.detach() for o in out], [o.requires_grad for o in out], x.grad, k.grad, node, seen


@pytest.mark.parametrize("x_grad,k_grad", [(True, True), (True, False), (False, True), (False, False)])
@pytest.mark.parametrize("hooks", [False, True])
def test_same_as_apply(x_grad, k_grad, hooks):
    a = _results(_Scaled.apply, x_grad, k_grad, hooks)
    b = _results(lambda *args: eager.apply(_Scaled, *args), x_grad, k_grad, hooks)
    for p, q in zip(a[0], b[0]):
        assert torch.equal(p, q)
    assert a[1] == b[1] and a[4:] == b[4:]
    for p, q in zip(a[2:4], b[2:4]):
        assert (p is None) == (q is None) and (p is None or torch.equal(p, q))


def test_no_grad_and_inference_mode():
    for mode in (torch.no_grad, torch.inference_mode):
        with mode():
            out = eager.apply(_Scaled, torch.ones(3, requires_grad=True), torch.tensor(2.0), (1.0,))
        assert not out[0].requires_grad and torch.equal(out[0], torch.full((3,), 2.0))


def test_forward_mode_is_refused_as_before():
    import torch.autograd.forward_ad as fwd

    for apply in (_Scaled.apply, lambda *args: eager.apply(_Scaled, *args)):
        with fwd.dual_level(), pytest.raises(RuntimeError):
            apply(fwd.make_dual(torch.ones(3), torch.ones(3)), torch.tensor(2.0), (1.0,))


def test_function_transforms():
    f = lambda apply: torch.func.grad(lambda x: apply(x, torch.tensor(2.0), (3.0,))[0].sum())(torch.ones(4))
    assert torch.equal(f(_Scaled.apply), f(lambda *args: eager.apply(_Scaled, *args)))


def test_second_derivative():
    x = torch.ones(3, requires_grad=True)
    grads = []
    for apply in (_Scaled.apply, lambda *args: eager.apply(_Scaled, *args)):
        k = torch.tensor(2.0, requires_grad=True)
        (g,) = torch.autograd.grad(apply(x, k, (3.0,))[0].sum(), x, create_graph=True)
        grads.append(torch.autograd.grad(g.sum(), k)[0])
    assert torch.equal(*grads)


def test_trace_keeps_the_function():
    traced = torch.jit.trace(lambda x: eager.apply(_Scaled, x, torch.tensor(2.0), (1.0,))[0], (torch.ones(3),))
    assert torch.equal(traced(torch.full((3,), 4.0)), torch.full((3,), 8.0))
