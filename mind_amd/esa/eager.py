"""When a call may go straight to the kernels.

A kernel entry takes device pointers, so whatever has to see the call as an
operation (torch.compile, make_fx and other dispatch modes, vmap / jvp, jit
tracing, tensor subclasses such as fake tensors) must get the registered
operator or the autograd function.  ``plain`` says that nothing of the kind is
active; the call can then skip their host cost: a registered operator's
dispatch takes about 140 us per forward and backward here, an autograd
function's about 6 us, the kernels of a small batch 10-40 us.
"""
from __future__ import annotations

import torch
from torch.autograd import forward_ad

_PLAIN = (torch.Tensor, torch.nn.Parameter)
_dispatch_modes = torch._C._len_torch_dispatch_stack
_function_modes = torch._C._len_torch_function_stack
_transforms = torch._C._functorch.peek_interpreter_stack
_tracing = torch._C._get_tracing_state


def plain(*args) -> bool:
    """True in ordinary eager execution on ordinary tensors (arguments that are no tensors are not looked at)."""
    if (torch.compiler.is_compiling() or _dispatch_modes() or _function_modes() or _transforms() is not None
            or forward_ad._current_level >= 0 or _tracing() is not None):
        return False
    return all(type(a) in _PLAIN or not isinstance(a, torch.Tensor) for a in args)


def records(*args) -> bool:
    """Whether autograd would record an operation on these arguments."""
    return torch.is_grad_enabled() and any(isinstance(a, torch.Tensor) and a.requires_grad for a in args)


class Unrecorded:
    """The context of a forward that autograd does not record: nothing is kept."""

    needs_input_grad = ()

    def save_for_backward(self, *tensors):
        pass

    def set_materialize_grads(self, value):
        pass

    def mark_non_differentiable(self, *tensors):
        pass


def call(function, *args):
    """``function.apply(*args)`` of an autograd function; its forward alone where nothing records or traces it."""
    if not records(*args) and plain(*args):
        return function.forward(Unrecorded(), *args)
    return function.apply(*args)
