"""Projections of the models: torch.nn.Linear whose products without a gradient go through `ops.linear`."""
from __future__ import annotations

import torch
import torch.nn as nn
import torch.nn.functional as F
from torch.autograd import forward_ad
from torch.nn.modules import module as nn_module

from . import ops


def _plain(x, weight) -> bool:
    """Nothing watches or rewrites torch's operations here: no gradient of either mode, no autocast, no tracing, compiling or vmap, no subclass
    of a tensor."""
    return (type(x) is torch.Tensor and type(weight) in (torch.Tensor, nn.Parameter) and not torch.compiler.is_compiling()
            and not torch.is_grad_enabled() and x.is_cuda and forward_ad._current_level < 0 and not torch.is_autocast_enabled("cuda")
            and not torch._C._is_tracing() and not torch._C._functorch.is_functorch_wrapped_tensor(x)
            and torch._C._len_torch_dispatch_stack() == 0 and torch._C._len_torch_function_stack() == 0)


def linear(x, weight, bias=None):
    return ops.linear(x, weight, bias) if _plain(x, weight) else F.linear(x, weight, bias)


class Linear(nn.Linear):
    def forward(self, x):
        return linear(x, self.weight, self.bias)


def swiglu(fc: nn.Linear, x):
    """`ops.swiglu` of fc(x), in one launch where nothing wants to see what lies between or has put a forward of its own into fc."""
    if (type(fc) is Linear and "forward" not in fc.__dict__ and not (fc._forward_hooks or fc._forward_pre_hooks or nn_module._global_forward_hooks
                                    or nn_module._global_forward_pre_hooks) and _plain(x, fc.weight)):
        return ops.swiglu(x, fc.weight, fc.bias)
    return ops.swiglu(fc(x))
