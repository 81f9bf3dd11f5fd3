"""Projections of the models: torch.nn.Linear whose products without a gradient go through `ops.linear`."""
from __future__ import annotations

import torch
import torch.nn as nn
import torch.nn.functional as F
from torch.autograd import forward_ad
from torch.nn.modules import module as nn_module

from . import ops


def _questions(c=torch._C, ad=forward_ad):
    """What tells whether torch's operations are watched, and has no public name; None where a torch build lacks one of them."""
    try:
        ad._current_level
        return c._functorch.peek_interpreter_stack, c._len_torch_dispatch_stack, c._len_torch_function_stack
    except AttributeError:
        return None


_QUESTIONS = _questions()

# Names of this module for what a model asks 119 times a prompt: with them, and the channels by the module, 2.2 us a projection for 3.0.
_is_tracing = getattr(torch._C, "_is_tracing", torch.jit.is_tracing)
_is_grad_enabled, _is_compiling, _is_autocast_enabled = torch.is_grad_enabled, torch.compiler.is_compiling, torch.is_autocast_enabled
_BF16, _STRIDED, _TENSORS = torch.bfloat16, torch.strided, (torch.Tensor, nn.Parameter)


def _beyond(x, weight, K=None) -> bool:
    """Torch's own for certain: a gradient, a compiler or a trace wants it, it is not in bf16 or there are too many rows.  Asked in front of
    everything else, for what the library takes waits for the host as well (the 360M model, 1 x 600 tokens: 4.8 ms, 5.1 where each projection's form
    was looked up first)."""
    if _is_grad_enabled() or _is_compiling() or _is_tracing() or x.dtype is not _BF16:
        return True
    if K is None:
        K = weight.size(-1)
    return x.numel() > ops.linear_max_rows(K) * K


def _watched() -> bool:
    """Something else watches or rewrites torch's operations: autocast (of the GPU), forward mode, vmap (of which the weight or the bias may be mapped
    and x not), a mode.  Or it cannot be told."""
    if _QUESTIONS is None or forward_ad._current_level >= 0 or _is_autocast_enabled():
        return True
    transform, dispatch_modes, function_modes = _QUESTIONS
    return transform() is not None or dispatch_modes() > 0 or function_modes() > 0


def _ordinary(t) -> bool:
    """A tensor with rows: no subclass, not sparse, not nested."""
    return type(t) in _TENSORS and t.layout is _STRIDED and not t.is_nested


def _plain(x, weight, bias) -> bool:
    """Tensors on the GPU, and nothing that watches (behind `_beyond`)."""
    return _ordinary(x) and _ordinary(weight) and (bias is None or _ordinary(bias)) and x.is_cuda and not _watched()


def linear(x, weight, bias=None):
    if _beyond(x, weight) or not _plain(x, weight, bias):
        return F.linear(x, weight, bias)
    return ops.linear(x, weight, bias)


def linear_like(x, K: int):
    """`linear` for several products of as many rows of K channels as x has, whose sizes are then asked once where torch has them."""
    return F.linear if _beyond(x, None, K) else linear


class Linear(nn.Linear):
    def _operands(self):
        own = self._parameters  # (`self.weight` looks through Module.__getattr__ first, half a microsecond)
        try:
            return own["weight"], own["bias"]
        except KeyError:  # (something else stands in for them)
            return self.weight, self.bias

    def forward(self, x):
        if torch.jit.is_scripting():
            return F.linear(x, self.weight, self.bias)
        weight, bias = self._operands()
        if _beyond(x, weight, self.in_features) or not _plain(x, weight, bias):
            return F.linear(x, weight, bias)
        return ops.linear(x, weight, bias)


def _alone(fc: Linear) -> bool:
    """A projection without hooks, of which nothing has put a forward of its own into it."""
    return "forward" not in fc.__dict__ and not (
        fc._forward_hooks or fc._forward_pre_hooks or nn_module._global_forward_hooks or nn_module._global_forward_pre_hooks)


def swiglu(fc: nn.Linear, x):
    """`ops.swiglu` of fc(x), in one launch where nothing wants to see what lies between."""
    if type(fc) is Linear and not _beyond(x, None, fc.in_features) and _alone(fc):
        weight, bias = fc._operands()
        if _plain(x, weight, bias):
            return ops.swiglu(x, weight, bias)
    return ops.swiglu(fc(x))
