"""Plain bfloat16 linears of the stateful decoders: nn.Linear to everything that holds, converts or hooks it, with the streamed-weights
kernel behind the few rows of a decode step."""

import torch.nn as nn
import torch.nn.functional as F
from torch import Tensor
from torch.nn.modules import module as _module

from . import seq_ops


class DecodeLinear(nn.Linear):
    def forward(self, x: Tensor) -> Tensor:
        weight, bias = self.weight, self.bias
        # the count first: the linears of short prompts are bound by what the host does for each of them
        if x.numel() <= seq_ops.STREAMED_ROWS * self.in_features and bias is None and seq_ops.linear_streams(x, weight):
            return seq_ops.linear(x, weight)
        return F.linear(x, weight, bias)


def unwatched(module: nn.Module) -> bool:
    """True where calling the module is no more than its class's forward: no forward of the instance's own, no hooks, not compiled."""
    return not ("forward" in module.__dict__ or module._compiled_call_impl is not None or module._forward_hooks or module._forward_pre_hooks
                or module._backward_hooks or module._backward_pre_hooks or _module._global_forward_hooks or _module._global_forward_pre_hooks
                or _module._global_backward_hooks or _module._global_backward_pre_hooks)


def fusable(lin: nn.Module, x: Tensor) -> bool:
    """True where lin(x) may be computed together with what follows it: the module itself (not a replacement), nobody watching its
    call, and an input that its kernel takes."""
    return (type(lin) is DecodeLinear and x.numel() <= seq_ops.STREAMED_ROWS * lin.in_features and lin.bias is None and seq_ops.linear_streams(x, lin.weight)
            and unwatched(lin))
