"""The base of this package's autograd Functions."""
import torch

from ._lib import host

_apply = torch.autograd.Function.apply.__func__


class Function(torch.autograd.Function):
    """``apply`` straight to torch's binding where ``torch.autograd.Function.apply`` has nothing to add: no functorch
    transform, no tensor that one has left wrapped (its own look at that takes 2 us a call), and no ``torch.compile``, which
    knows that function and not the binding."""

    @classmethod
    def apply(cls, *args):
        if torch.compiler.is_compiling() or torch._C._are_functorch_transforms_active() or not host.unwrapped(*args):
            return _apply(cls, *args)
        return super(torch.autograd.Function, cls).apply(*args)
