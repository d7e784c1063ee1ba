"""Which Llama-layer calls keep torch's operators: everything that watches their input (layer._unwatched) or
their weights (layer._plain_weight)."""

import torch

from apple_amd.layer import _plain_weight, _unwatched


def test_unwatched():
    x = torch.zeros(1, 2, 4)
    assert _unwatched(x)
    g = torch.zeros(1, 2, 4, requires_grad=True)
    assert not _unwatched(g)
    with torch.no_grad():
        assert _unwatched(g)
    seen = []
    torch.func.vmap(lambda t: seen.append(_unwatched(t)) or t)(x)
    torch.func.grad(lambda t: seen.append(_unwatched(t)) or t.sum())(x)
    torch.func.jvp(lambda t: seen.append(_unwatched(t)) or t, (x,), (x,))
    with torch.autograd.forward_ad.dual_level():
        seen.append(_unwatched(torch.autograd.forward_ad.make_dual(x, x)))
    torch.jit.trace(lambda t: seen.append(_unwatched(t)) or t + 1, (x,), check_trace=False)
    from torch.utils.flop_counter import FlopCounterMode

    with FlopCounterMode(display=False):
        seen.append(_unwatched(x))

    class Mode(torch.overrides.TorchFunctionMode):
        def __torch_function__(self, f, types, args=(), kwargs=None):
            return f(*args, **(kwargs or {}))

    with Mode():
        seen.append(_unwatched(x))

    class Sub(torch.Tensor):
        pass

    seen.append(_unwatched(x.as_subclass(Sub)))
    assert seen and not any(seen), seen


def test_weights_under_transforms():
    """torch.func over a layer's weights hands it wrapped tensors without storage beside a plain input."""
    cpu = torch.device("cpu")
    w = torch.zeros(4, 8)
    assert _plain_weight(w, cpu) and _plain_weight(torch.nn.Parameter(w, requires_grad=False), cpu)
    seen = []
    look = lambda t: seen.append(_plain_weight(t, cpu)) or t * 1.0
    torch.func.vmap(look)(torch.zeros(3, 4, 8))
    torch.func.grad(lambda t: look(t).sum())(w)
    torch.func.jvp(look, (w,), (w,))
    torch.func.vjp(look, w)
    layer = torch.nn.Linear(8, 4, bias=False)
    layer.forward = lambda x: x @ look(layer._parameters["weight"]).t()
    x = torch.zeros(1, 8)
    torch.func.grad(lambda t: torch.func.functional_call(layer, {"weight": t}, (x,)).sum())(w)
    seen += [_plain_weight(torch.zeros(4, 8, requires_grad=True), cpu), _plain_weight(w.double(), cpu),
             _plain_weight(w.t(), cpu), _plain_weight(torch.zeros(33)[1:], cpu)]
    assert len(seen) == 9 and not any(seen), seen
    with torch.no_grad():
        assert _plain_weight(torch.zeros(4, 8, requires_grad=True), cpu)
