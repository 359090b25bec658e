"""The base of this package's autograd Functions."""
import torch

from ._lib import host


class Function(torch.autograd.Function):
    """``apply`` straight to torch's binding where ``torch.autograd.Function.apply`` has nothing to add: no functorch
    transform, and no tensor that one has left wrapped (its own look at that takes 2 us a call)."""

    @classmethod
    def apply(cls, *args):
        if not torch._C._are_functorch_transforms_active() and host.unwrapped(*args):
            return super(torch.autograd.Function, cls).apply(*args)
        return super().apply(*args)
