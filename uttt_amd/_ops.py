"""torch.library registrations of this package's C-ABI calls (namespace
`uttt_hip`), each with a fake implementation that gives its outputs' shapes
and dtypes, so that torch.compile traces the drop-in ops into its graph
instead of breaking the graph at every kernel call.

`traced_op(name, fake)` registers a function as torch.ops.uttt_hip.<name>
and returns a wrapper that calls the registered op while torch.compile
traces, and the function itself otherwise (eager calls skip the dispatcher).
"""
from __future__ import annotations

import functools

import torch
from torch._C._functorch import is_dead_tensor_wrapper
from torch._functorch.utils import unwrap_dead_wrappers
from torch.autograd import forward_ad


def traced_op(name, fake, mutates_args=()):
    def deco(fn):
        op = torch.library.custom_op(f"uttt_hip::{name}", fn, mutates_args=mutates_args)
        op.register_fake(fake)

        @functools.wraps(fn)
        def call(*args, **kwargs):
            if torch.compiler.is_compiling():
                return op(*args, **kwargs)
            return fn(*args, **kwargs)

        call.op = op
        return call

    return deco


class _NoGraph:
    """The ctx of a forward whose graph nobody keeps."""

    def save_for_backward(self, *tensors):
        pass

    def mark_non_differentiable(self, *tensors):
        pass


def run_function(fn, *args):
    """fn.apply(*args) of a torch.autograd.Function, or its forward alone where
    nothing could see the difference: gradients are off and neither
    torch.compile, jit tracing, a functorch transform nor a forward-mode level
    is active (under which apply records, refuses or transforms the call).
    A forward that hands an input through returns it as it is, where apply
    returns an alias: its caller makes one (permute_with_expert_mask).
    apply costs 5 to 8 us of host time per call; a routed read without
    gradients, three of them, is paced by its host time (88 us against 61 on
    the GPU for 16 384 tokens of 192 over 48 experts)."""
    if (torch.is_grad_enabled() or torch.compiler.is_compiling()
            or torch._C._are_functorch_transforms_active()
            or torch._C._get_tracing_state() is not None or forward_ad._current_level >= 0):
        return fn.apply(*args)
    try:
        return fn.forward(_NoGraph(), *args)
    except RuntimeError:
        # a tensor that outlived its functorch transform is a shell without an
        # address around the real one, which apply hands on
        if not any(isinstance(a, torch.Tensor) and is_dead_tensor_wrapper(a) for a in args):
            raise
    return fn.forward(_NoGraph(), *unwrap_dead_wrappers(args))


def none_if_empty(t):
    """Optional outputs travel through the ops as 0-element tensors."""
    return None if t is None or t.numel() == 0 else t


def empty_like_dev(ref, *shape, dtype=None):
    return ref.new_empty(shape, dtype=ref.dtype if dtype is None else dtype)
