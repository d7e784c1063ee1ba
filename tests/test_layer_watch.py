"""Which Llama-layer calls keep torch's operators (layer._unwatched): everything that watches them."""

import torch

from apple_amd.layer import _unwatched


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
