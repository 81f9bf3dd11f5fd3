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
        return c._is_tracing, c._functorch.peek_interpreter_stack, c._len_torch_dispatch_stack, c._len_torch_function_stack
    except AttributeError:
        return None


_QUESTIONS = _questions()


def _watched() -> bool:
    """Something watches or rewrites torch's operations here: a gradient of either mode, autocast, tracing, compiling, vmap (of which the weight or
    the bias may be mapped and x not), a mode.  Or it cannot be told."""
    if torch.is_grad_enabled() or _QUESTIONS is None or torch.compiler.is_compiling() or torch.is_autocast_enabled("cuda"):
        return True
    tracing, transform, dispatch_modes, function_modes = _QUESTIONS
    return forward_ad._current_level >= 0 or tracing() or transform() is not None or dispatch_modes() > 0 or function_modes() > 0


def _ordinary(t) -> bool:
    """A tensor with rows: no subclass, not sparse, not nested."""
    return type(t) in (torch.Tensor, nn.Parameter) and t.layout is torch.strided and not t.is_nested


def _plain(x, weight, bias) -> bool:
    """Tensors on the GPU, and nothing that watches."""
    return _ordinary(x) and _ordinary(weight) and (bias is None or _ordinary(bias)) and x.is_cuda and not _watched()


def linear(x, weight, bias=None):
    return ops.linear(x, weight, bias) if _plain(x, weight, bias) else F.linear(x, weight, bias)


class Linear(nn.Linear):
    def forward(self, x):
        if torch.jit.is_scripting():
            return F.linear(x, self.weight, self.bias)
        return linear(x, self.weight, self.bias)


def swiglu(fc: nn.Linear, x):
    """`ops.swiglu` of fc(x), in one launch where nothing wants to see what lies between or has put a forward of its own into fc."""
    if (type(fc) is Linear and "forward" not in fc.__dict__ and not (fc._forward_hooks or fc._forward_pre_hooks or nn_module._global_forward_hooks
                                    or nn_module._global_forward_pre_hooks) and _plain(x, fc.weight, fc.bias)):
        return ops.swiglu(x, fc.weight, fc.bias)
    return ops.swiglu(fc(x))
