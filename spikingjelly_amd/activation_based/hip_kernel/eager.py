"""Eager application of the autograd functions of the fused chains."""

from __future__ import annotations

import torch

_twins: dict = {}


def _twin(function):
    """The same forward, context and backward with the context as the forward's first argument."""
    def forward(ctx, *args):
        output = function.forward(*args)
        function.setup_context(ctx, args, output)
        return output

    twin = type(function.__name__, (torch.autograd.Function,),
                {"__module__": function.__module__, "__doc__": function.__doc__, "forward": staticmethod(forward),
                 "backward": staticmethod(function.backward)})
    _twins[function] = twin
    return twin


def apply(function, *args):
    """``function.apply(*args)`` with every argument of its forward given by position.

    A function that has a ``setup_context`` gets its arguments bound to the signature of its forward on each call, 25 to 35 us
    of host time for the 9 to 12 arguments of a chain; a forward that takes the context itself is called as it is.  Function
    transforms ask for the separate context and keep it, a traced call keeps the function whose name the trace shows.  Both ways in
    turn in one process: attention block [4, 1, 384, 196] in evaluation mode, two calls, 263 -> 215 us; training step at
    [4, 2, 256, 64], two calls, 741 -> 667; convolution block [4, 2, 192, 49] -> 384, training step, one call, 366 -> 336."""
    if torch._C._are_functorch_transforms_active() or torch.jit.is_tracing():
        return function.apply(*args)
    return (_twins.get(function) or _twin(function)).apply(*args)
