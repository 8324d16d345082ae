"""Bedalorn: a pre-norm decoder of wkv and latent-attention layers with dense or
mixture-of-experts feed-forwards, part of whose layers run several times.

Layer:  x <- x + mixer(norm1(x));  x <- x + ff(norm2(x)).
Pass t of the repeated layers:  x <- W_in [x; x0] + step_t  ahead of its first.

The residual x is 32-bit; a sublayer's update of it waits for the next norm's
kernel.  W_in is kept as its two halves, so what it does to the embedding x0 is
computed once for all passes; both products stay in 32-bit.
"""
from __future__ import annotations

import copy
from dataclasses import dataclass, field

import torch
import torch.nn as nn
import torch.nn.functional as F

from .. import ops
from .feedforward import FEED_FORWARDS
from .mixers import SUBLAYER_MIXERS


@dataclass
class BedalornConfig:
    vocab_size: int
    hidden_size: int
    layers: list = field(default_factory=list)   # {"type", "mixer", "mlp"} each
    loop: dict | None = None                     # {"start", "stop", "times"}
    logit_scale: float = 1.0
    norm_eps: float = 1e-5
    dtype: str = "bfloat16"

    def __post_init__(self):
        for layer in self.layers:
            if layer["type"] not in SUBLAYER_MIXERS:
                raise ValueError(f"unknown mixer {layer['type']!r}; "
                                 f"have {sorted(SUBLAYER_MIXERS)}")
            mlp = layer.get("mlp")
            if mlp is not None and mlp["kind"] not in FEED_FORWARDS:
                raise ValueError(f"unknown feed-forward {mlp['kind']!r}; "
                                 f"have {sorted(FEED_FORWARDS)}")
        if self.loop and not 0 <= self.loop["start"] <= self.loop["stop"] <= len(self.layers):
            raise ValueError(f"loop {self.loop} of {len(self.layers)} layers")

    @classmethod
    def from_json(cls, c: dict, tensors: dict, **overrides) -> "BedalornConfig":
        """The rank of a wkv layer's decay is the checkpoint tensors' alone."""
        layers = copy.deepcopy(c["layers"])
        for i, layer in enumerate(layers):
            name = f"l{i}.mix.w1"
            if layer["type"] == "wkv" and name in tensors:
                layer["mixer"]["decay_rank"] = tensors[name].shape[0]
        d = dict(vocab_size=c["vocab"], hidden_size=c["width"], layers=layers,
                 loop=c.get("loop"), logit_scale=c["logit_scale"], norm_eps=c["norm"]["eps"])
        d.update(overrides)
        return cls(**d)

    @property
    def num_layers(self) -> int:
        return len(self.layers)

    def plan(self) -> list:
        """What a forward runs in order: ("pass", t) where pass t of the
        repeated layers starts, ("layer", i)."""
        n = len(self.layers)
        loop = self.loop or dict(start=n, stop=n, times=0)
        steps = [("layer", i) for i in range(loop["start"])]
        for t in range(loop["times"]):
            steps.append(("pass", t))
            steps += [("layer", i) for i in range(loop["start"], loop["stop"])]
        return steps + [("layer", i) for i in range(loop["stop"], n)]

    def cache_layers(self) -> list:
        """One entry per layer run: every pass keeps its own."""
        with torch.device("meta"):
            specs = [SUBLAYER_MIXERS[l["type"]](self.hidden_size, l["mixer"],
                                                self.norm_eps).cache_spec for l in self.layers]
        return [specs[i] for kind, i in self.plan() if kind == "layer"]


class SequentialBlock(nn.Module):
    def __init__(self, cfg: BedalornConfig, layer: dict):
        super().__init__()
        W = cfg.hidden_size
        self.norm1 = nn.Parameter(torch.empty(W))
        self.mixer = SUBLAYER_MIXERS[layer["type"]](W, layer["mixer"], cfg.norm_eps)
        mlp = layer.get("mlp")
        self.mlp = None
        if mlp is not None:
            self.norm2 = nn.Parameter(torch.empty(W))
            self.mlp = FEED_FORWARDS[mlp["kind"]](W, mlp)

    def load(self, take) -> None:
        W = (self.norm1.shape[0],)
        self.norm1.copy_(take("norm1", W))
        self.mixer.load(lambda name, shape: take("mix." + name, shape))
        if self.mlp is not None:
            self.norm2.copy_(take("norm2", W))
            self.mlp.load(lambda name, shape: take("mlp." + name, shape))

    def forward(self, norm, pending: dict, ctx, cache) -> torch.Tensor:
        """norm(weight, **pending) updates the residual and norms it.  Returns
        the update that is left pending."""
        delta = self.mixer(norm(self.norm1, **pending), ctx, cache)
        return delta if self.mlp is None else self.mlp(norm(self.norm2, delta=delta))


class BedalornLM(nn.Module):
    """Served through SamplerEngine like CausalLM: forward(ids, ctx) returns
    final normed hidden states, logits() applies the (tied) head."""

    extensions = ("_serve",)            # HIP extensions its forward needs
    kv_cache_dtypes = ("bf16",)         # "bf16" = pages in the model's dtype
    packed_prefill = False              # prompts run through step portions

    def __init__(self, cfg: BedalornConfig, init: bool = True):
        super().__init__()
        self.cfg = cfg
        W = cfg.hidden_size
        self.plan = cfg.plan()
        self.embed = nn.Parameter(torch.empty(cfg.vocab_size, W))
        self.layers = nn.ModuleList(SequentialBlock(cfg, l) for l in cfg.layers)
        self.norm = nn.Parameter(torch.empty(W))
        if cfg.loop:
            self.in_x = nn.Parameter(torch.empty(W, W))     # W_in's half for x
            self.in_x0 = nn.Parameter(torch.empty(W, W))    # and for the embedding
            self.step = nn.Parameter(torch.empty(cfg.loop["times"], W))
        if init:
            self._load(lambda name, shape: torch.randn(shape, dtype=self.norm.dtype,
                                                       device=self.norm.device) * 0.02)

    @property
    def lm_head_weight(self) -> torch.Tensor:
        return self.embed

    @torch.no_grad()
    def _load(self, take) -> None:
        """take(name, shape) -> tensor"""
        W = self.cfg.hidden_size
        self.embed.copy_(take("embed", (self.cfg.vocab_size, W)))
        self.norm.copy_(take("final.norm", (W,)))
        if self.cfg.loop:
            w = take("loop.in", (W, 2 * W))
            self.in_x.copy_(w[:, :W])
            self.in_x0.copy_(w[:, W:])
            self.step.copy_(take("loop.step", (self.cfg.loop["times"], W)))
        for i, b in enumerate(self.layers):
            b.load(lambda name, shape, i=i: take(f"l{i}.{name}", shape))

    def load(self, tensors: dict) -> None:
        used = set()

        def take(name, shape):
            if name not in tensors:
                raise KeyError(f"checkpoint is missing tensor {name!r}")
            if tuple(tensors[name].shape) != tuple(shape):
                raise ValueError(f"{name}: shape {tuple(tensors[name].shape)}, "
                                 f"expected {tuple(shape)}")
            used.add(name)
            return tensors[name]

        self._load(take)
        # a layer without a feed-forward has no use for its second norm
        used |= {f"l{i}.norm2" for i, b in enumerate(self.layers) if b.mlp is None}
        extra = sorted(set(tensors) - used)
        if extra:
            raise RuntimeError(f"unmapped checkpoint tensors: {extra[:8]}")

    def forward(self, input_ids: torch.Tensor, ctx) -> torch.Tensor:
        if ctx.mode not in ("step", "decode"):
            raise NotImplementedError(f"Bedalorn is served, not trained (mode {ctx.mode!r})")
        eps = self.cfg.norm_eps
        x = torch.empty(input_ids.shape[0], self.cfg.hidden_size, dtype=torch.float32,
                        device=input_ids.device)
        pending = dict(embed=self.embed, ids=input_ids)     # not in x yet

        def norm(weight, **update):
            return ops.residual_group_norm(x, weight, eps, offset=1.0, **update)

        into, run = None, 0
        if self.cfg.loop:
            x0 = F.embedding(input_ids, self.embed)
            into = linear_f32(x0, self.in_x0)
        for kind, i in self.plan:
            if kind == "pass":
                y = x0 if "ids" in pending else norm(None, **pending)
                x = linear_f32(y, self.in_x)
                pending = dict(add=into, bias=self.step[i])
                continue
            pending = dict(delta=self.layers[i](norm, pending, ctx, ctx.kv_caches[run]))
            if ctx.on_layer is not None:
                d = pending["delta"].float()
                ctx.on_layer(run, x + (d if d.dim() == 2 else d.sum(1)))
            run += 1
        return ops.residual_group_norm(x, self.norm, eps, offset=1.0,
                                       gain=self.cfg.logit_scale, **pending)

    def logits(self, hidden: torch.Tensor) -> torch.Tensor:
        """hidden carries the logit scale."""
        return ops.linear(hidden, self.embed)


def linear_f32(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """x w^T, the 32-bit sums as they are."""
    if x.is_cuda and x.dtype != torch.float32:
        return torch.mm(x, w.t(), out_dtype=torch.float32)
    return F.linear(x.float(), w.float())
