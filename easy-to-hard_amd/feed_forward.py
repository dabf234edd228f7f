"""Feed-forward sublayers: squared ReLU, and a mixture of such experts."""

from typing import Optional, Tuple

import torch
import torch.nn as nn
from torch import Tensor

from . import seq_ops
from .linear import DecodeLinear, fusable, unwatched


class SquaredReluFF(nn.Module):
    def __init__(self, width: int, hidden: int):
        super().__init__()
        self.up = DecodeLinear(width, hidden, bias=False)
        self.down = DecodeLinear(hidden, width, bias=False)

    def forward(self, h: Tensor, defer: bool = False) -> Tensor:
        """defer (a step whose next norm is seq_ops.norm_conv's): the result may come as float32 sums over slices of K, for that to add."""
        if fusable(self.up, h):
            y = seq_ops.linear(h, self.up.weight, seq_ops.ACT_SQUARE_RELU)
            sums = seq_ops.linear_sums(y, self.down.weight) if defer and fusable(self.down, y) else None
            return self.down(y) if sums is None else sums
        if type(self.up) is DecodeLinear and self.up.bias is None and unwatched(self.up) and seq_ops.linear_rows_pay(h, self.up.weight, seq_ops.ACT_SQUARE_RELU):
            return self.down(seq_ops.linear_rows(h, self.up.weight, seq_ops.ACT_SQUARE_RELU))
        return self.down(seq_ops.square_relu_(self.up(h)))


class ExpertMixture(nn.Module):
    """Squared-ReLU experts of which every token uses the `top` ones with the largest router logits, weighted by the softmax over
    those logits, and an optional shared expert that every token uses.

    `forward` returns the parts of the sum: the shared expert's rows (or None), the chosen experts' rows [rows * top, width] and
    their weights [rows, top]; the pass that normalises the sum (seq_ops.norm_conv) also forms it.  The shared expert's linears
    are ordinary modules, so a QuantHandler can replace them; the experts are kept as two stacks."""

    STEP_ROWS = 64  # up to here the shared expert runs inside the experts' launches (they read weights, not activations)

    def __init__(self, width: int, experts: int, top: int, hidden: int, shared_hidden: Optional[int]):
        super().__init__()
        self.top = top
        self.router = nn.Parameter(torch.zeros((experts, width)), requires_grad=False)
        self.router_bias = nn.Parameter(torch.zeros((experts,), dtype=torch.float32), requires_grad=False)
        self.up = nn.Parameter(torch.zeros((experts, hidden, width)), requires_grad=False)
        self.down = nn.Parameter(torch.zeros((experts, width, hidden)), requires_grad=False)
        self.shared = SquaredReluFF(width, shared_hidden) if shared_hidden else None

    def forward(self, h: Tensor) -> Tuple[Optional[Tensor], Tensor, Tensor]:
        chosen, weights = seq_ops.route(h, self.router, self.router_bias, self.top)
        if self.shared is not None and h.shape[0] <= self.STEP_ROWS and self._shared_joins():
            out, shared = seq_ops.experts(h, chosen, self.up, self.down, self.shared.up.weight, self.shared.down.weight)
            return shared, out, weights
        out, _ = seq_ops.experts(h, chosen, self.up, self.down)
        return (None if self.shared is None else self.shared(h)), out, weights

    def _shared_joins(self) -> bool:
        """the shared expert is the modules built here, and nobody watches their calls"""
        linears = (self.shared.up, self.shared.down)
        return all(type(m) in (nn.Linear, DecodeLinear) for m in linears) and unwatched(self.shared) and all(unwatched(m) for m in linears)

    def from_checkpoint(self, get, prefix: str, linear_dtype) -> dict:
        n = self.router.shape[0]
        sd = {"router": get(prefix + ".router").to(linear_dtype), "router_bias": get(prefix + ".router.b").float()}
        for name in ("up", "down"):
            sd[name] = torch.stack([get(f"{prefix}.e{i}.{name}").to(linear_dtype) for i in range(n)])
            if self.shared is not None:
                sd[f"shared.{name}.weight"] = get(f"{prefix}.shared.{name}").to(linear_dtype)
        return sd
