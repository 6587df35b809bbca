"""Transforms of a call that a hand-made C++ node does not stand for: refused, or taken by a path that they see, as by the
autograd.Functions in Python.  The layers around the attention here, on the CPU; tests/test_gpu_host_path.py has the attention."""
import pytest
import torch
from torch import nn

from evoformer_triton_amd import block


def _calls(requires_grad=True):
    g = torch.Generator().manual_seed(8)
    layer = nn.Linear(16, 8).requires_grad_(requires_grad)
    ws = [torch.randn((8, 16), generator=g, requires_grad=requires_grad) for _ in range(4)]
    bg = torch.randn((8,), generator=g, requires_grad=requires_grad)
    return {"linear": lambda x: block._linear(layer, x), "stacked": lambda x: block._StackedProjection.apply(x, bg, *ws)}


@pytest.mark.parametrize("name", ["linear", "stacked"])
def test_functorch_transforms_are_refused(name):
    call, x = _calls()[name], torch.randn(3, 5, 16)
    with pytest.raises(RuntimeError, match="setup_context"):
        torch.vmap(call)(x)
    with pytest.raises(RuntimeError, match="setup_context"):
        torch.func.grad(lambda t: call(t).sum())(x)
    assert call(x).grad_fn is not None


@pytest.mark.parametrize("name", ["linear", "stacked"])
def test_a_dispatch_mode_sees_the_layers_and_changes_nothing(name):
    from torch.utils._python_dispatch import TorchDispatchMode
    call, x = _calls()[name], torch.randn(3, 5, 16)
    seen = []

    class Recorder(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(str(func))
            return func(*args, **(kwargs or {}))

    want = call(x)
    with Recorder():
        got = call(x)
    assert torch.equal(got, want) and any("mm" in f for f in seen)


@pytest.mark.parametrize("name", ["linear", "stacked"])
def test_a_forward_mode_tangent_is_refused_not_dropped(name):
    from torch.autograd import forward_ad
    call, x = _calls()[name], torch.randn(3, 5, 16)
    with forward_ad.dual_level():
        with pytest.raises(NotImplementedError, match="jvp|forward mode"):
            call(forward_ad.make_dual(x, torch.ones_like(x)))


def test_a_forward_mode_tangent_of_a_parameter_is_refused():
    from torch.autograd import forward_ad
    x = torch.randn(3, 5, 16)
    with forward_ad.dual_level():
        for part in ("weight", "bias"):
            layer = nn.Linear(16, 8)
            p = getattr(layer, part).detach()
            delattr(layer, part)
            setattr(layer, part, forward_ad.make_dual(p, torch.ones_like(p)))
            with pytest.raises(NotImplementedError, match="jvp|forward mode"):
                block._linear(layer, x)


@pytest.mark.parametrize("name", ["linear", "stacked"])
def test_a_traced_layer_computes_on_replay(name):
    call = _calls(requires_grad=False)[name]     # (the tracer takes what a call closes over as constants)
    traced = torch.jit.trace(call, (torch.randn(3, 5, 16),), check_trace=False)
    x = torch.randn(3, 5, 16)
    assert torch.equal(traced(x), call(x)) and "_Linear" in str(traced.inlined_graph)
