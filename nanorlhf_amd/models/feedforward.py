"""Feed-forward sublayers of the sequential-block models: h [T, W] in, the
residual's update out ([T, W], or [T, parts, W] whose parts are to be added)."""
from __future__ import annotations

import torch
import torch.nn as nn
import torch.nn.functional as F

from .. import ops
from .lora import project

ALIGN = 8


class SquaredReluMLP(nn.Module):
    def __init__(self, width: int, m: dict):
        super().__init__()
        self.ff = m["ff"]
        self.up = nn.Linear(width, self.ff, bias=False)
        self.down = nn.Linear(self.ff, width, bias=False)

    def load(self, take) -> None:
        W = self.up.in_features
        self.up.weight.copy_(take("up", (self.ff, W)))
        self.down.weight.copy_(take("down", (W, self.ff)))

    def forward(self, h):
        return project(self.down, ops.relu_squared_(project(self.up, h)))


class MixtureOfExperts(nn.Module):
    """`top` of `experts` gated feed-forwards per token, weighted by the softmax
    over the chosen logits.  The experts' widths are padded with zeros."""

    def __init__(self, width: int, m: dict):
        super().__init__()
        self.experts, self.top = m["router"]["experts"], m["router"]["top"]
        if not 1 <= self.top <= self.experts:
            raise ValueError(f"top {self.top} of {self.experts} experts")
        self.ff, self.width = m["expert"]["ff"], width
        ffp = -(-self.ff // ALIGN) * ALIGN
        self.router = nn.Parameter(torch.empty(self.experts, width))
        self.router_bias = nn.Parameter(torch.empty(self.experts))
        self.gate_up = nn.Parameter(torch.empty(self.experts, 2, ffp, width))
        self.down = nn.Parameter(torch.empty(self.experts, width, ffp))

    def load(self, take) -> None:
        W, ff = self.width, self.ff
        self.router.copy_(take("router", (self.experts, W)))
        self.router_bias.copy_(take("router.b", (self.experts,)))
        self.gate_up[:, :, ff:].zero_()
        self.down[:, :, ff:].zero_()
        for e in range(self.experts):
            self.gate_up[e, 0, :ff].copy_(take(f"e{e}.gate", (ff, W)))
            self.gate_up[e, 1, :ff].copy_(take(f"e{e}.up", (ff, W)))
            self.down[e, :, :ff].copy_(take(f"e{e}.down", (W, ff)))

    def forward(self, h):
        routing = ops.moe_route(h, self.router, self.router_bias, self.top)
        return ops.moe_experts(h, self.gate_up, self.down, routing)


FEED_FORWARDS = {"dense": SquaredReluMLP, "moe": MixtureOfExperts}
