"""MI355X-native Qwen2-architecture causal LM.

Replaces the reference's transformers Qwen2 + flash_attention_2 stack
(GRPO/grpo.py:218-224).  Design choices (MI355X-first, not a port):

  * packed varlen layout everywhere — no pad tokens reach compute; the
    collator packs, attention gets cu_seqlens (the reference instead builds
    pad masks in a local forward(), grpo_trainer.py:90-120);
  * hot ops route through nanorlhf_amd.ops (hand-written HIP on GPU);
  * plain projections of many rows stay torch.nn.functional.linear →
    rocBLAS/hipBLASLt, few rows take ops.linear's kernel;
  * the SAME module graph serves training, prefill and paged decode — the
    in-process sampler passes an AttnContext instead of booting a separate
    engine (deletes the reference's disk round trip, grpo_trainer.py:122-166).
"""
from __future__ import annotations

from dataclasses import dataclass, field
from typing import Callable, Optional

import torch
import torch.nn as nn
import torch.nn.functional as F

from .. import ops
from ..ops.linear import FEW_ROWS
from .config import ModelConfig, get_config
from .lora import plain_weight, project, unheard


@dataclass
class Portions:
    """The multi-token entries of an engine step, packed; every tensor is on
    the model's device and int32."""
    cu: torch.Tensor               # [B+1] first row of each portion
    seq_lens: torch.Tensor         # [B] tokens of the sequence, these included
    block_tables: torch.Tensor     # [B, P]
    row_seq: torch.Tensor          # [rows] portion of each row
    state_slots: torch.Tensor      # [B]
    fresh: torch.Tensor            # [B] 1 where the portion starts its sequence
    chunks: torch.Tensor           # [3, n] portion, first row, tokens (<= 64)
    chunk_first: torch.Tensor      # [B+1] first chunk of each portion
    max_q: int = 0                 # longest portion
    # the portions' whole contexts laid out one after the other, each from a
    # multiple of the chunk size
    ctx_first: Optional[torch.Tensor] = None     # [B+1] first row of each context
    keys: int = 0                  # rows of that layout
    pairs: int = 0                 # sum of tokens x context length


@dataclass
class AttnContext:
    """Per-forward attention routing info.

    "train" and "prefill" pack whole sequences (cu_seqlens); "decode" is one
    token of each sequence; "step" is one batch of n_decode single tokens
    followed by the tokens of `portions`, all over the cache."""
    mode: str                      # "train" | "prefill" | "decode" | "step"
    positions: torch.Tensor        # [T] int64 position ids
    cu_seqlens: Optional[torch.Tensor] = None   # [B+1] int32 (train/prefill)
    max_seqlen: int = 0
    # paged-KV fields (prefill writes, decode reads+writes)
    kv_caches: Optional[list] = None            # per layer (k_cache, v_cache)
    slots: Optional[torch.Tensor] = None        # [T] int64 flat slot ids
    block_tables: Optional[torch.Tensor] = None  # [B, P] int32 (decode)
    seq_lens: Optional[torch.Tensor] = None      # [B] int32 (decode)
    state_slots: Optional[torch.Tensor] = None   # [B] int32 (decode)
    causal: bool = True
    portions: Optional[Portions] = None
    on_layer: Optional[Callable] = None          # observer: (layer, residual stream)
    _angles: dict = field(default_factory=dict)

    @property
    def n_decode(self) -> int:
        """Single-token rows at the head of a "step" or "decode" batch."""
        return 0 if self.seq_lens is None else self.seq_lens.shape[0]

    def angles(self, rotation) -> torch.Tensor:
        """cos | sin rows of this batch's tokens, once per distinct rotation."""
        if rotation.key not in self._angles:
            self._angles[rotation.key] = rotation.angles(self.positions)
        return self._angles[rotation.key]


def dtype_of(cfg: ModelConfig):
    return getattr(torch, cfg.dtype)


class Attention(nn.Module):
    def __init__(self, cfg: ModelConfig, layer_idx: int):
        super().__init__()
        self.layer_idx = layer_idx
        self.num_heads = cfg.num_heads
        self.num_kv_heads = cfg.num_kv_heads
        self.head_dim = cfg.head_dim
        H = cfg.hidden_size
        self.q_size = cfg.num_heads * cfg.head_dim
        self.kv_size = cfg.num_kv_heads * cfg.head_dim
        # fused qkv projection: one GEMM instead of three (MI355X-first —
        # bigger N per launch; the reference's transformers Qwen2 keeps
        # separate q/k/v linears)
        self.qkv_proj = nn.Linear(H, self.q_size + 2 * self.kv_size, bias=cfg.qkv_bias)
        self.o_proj = nn.Linear(cfg.num_heads * cfg.head_dim, H, bias=False)
        self.scale = cfg.head_dim ** -0.5

    def forward(self, x: torch.Tensor, rope_table: torch.Tensor, ctx: AttnContext,
                parts: bool = False):
        T = x.shape[0]
        cached = ctx.mode != "train" and ctx.kv_caches is not None
        qkv = project(self.qkv_proj, x, parts=cached)
        if cached:
            q, k, v = ops.qkv_rope_append(qkv, rope_table, ctx.positions, self.num_heads,
                                          ctx.slots, *ctx.kv_caches[self.layer_idx],
                                          want_kv=ctx.mode not in ("decode", "step"),
                                          bias=getattr(self.qkv_proj, "bias", None))
        else:
            q, k, v = ops.qkv_rope(qkv, rope_table, ctx.positions, self.num_heads,
                                   self.num_kv_heads)

        if ctx.mode == "decode":
            o = ops.paged_attn_decode(q, *ctx.kv_caches[self.layer_idx],
                                      ctx.block_tables, ctx.seq_lens, self.scale)
        elif ctx.mode == "step":
            o = torch.empty(T, self.q_size, dtype=q.dtype, device=q.device)
            ops.paged_attn(q, *ctx.kv_caches[self.layer_idx], ctx, o, self.scale)
        else:
            o = ops.flash_attn_varlen(q, k, v, ctx.cu_seqlens, ctx.max_seqlen,
                                      self.scale, causal=ctx.causal)
        return project(self.o_proj, o.reshape(T, -1),
                       parts and getattr(self.o_proj, "bias", None) is None)


class MLP(nn.Module):
    def __init__(self, cfg: ModelConfig):
        super().__init__()
        self.gate_up_proj = nn.Linear(cfg.hidden_size, 2 * cfg.intermediate_size, bias=False)
        self.down_proj = nn.Linear(cfg.intermediate_size, cfg.hidden_size, bias=False)

    def forward(self, x, parts: bool = False):
        w = plain_weight(self.gate_up_proj)
        if w is None or self.gate_up_proj.bias is not None:
            act = ops.swiglu(self.gate_up_proj(x))
        else:
            act = ops.linear_swiglu(x, w)
        return project(self.down_proj, act,
                       parts and getattr(self.down_proj, "bias", None) is None)


class RMSNorm(nn.Module):
    def __init__(self, hidden_size: int, eps: float):
        super().__init__()
        self.weight = nn.Parameter(torch.ones(hidden_size))
        self.eps = eps

    def forward(self, x):
        return ops.rms_norm(x, self.weight, self.eps)


def _plain(m: nn.Module, cls: type) -> bool:
    """Whether a call of this module is what this file says of `cls`, and nobody watches it."""
    return (type(m) is cls and cls.forward is _FORWARDS[cls] and "forward" not in m.__dict__
            and m._compiled_call_impl is None and unheard(m))


def _few(rows: int) -> bool:
    """Whether a projection of so many rows may come in parts at all."""
    return rows <= FEW_ROWS and not torch.is_grad_enabled()


def _parts(m: nn.Module, cls: type) -> dict:
    """What lets a module that nobody watches return parts."""
    return dict(parts=True) if _plain(m, cls) else {}


class Block(nn.Module):
    def __init__(self, cfg: ModelConfig, layer_idx: int):
        super().__init__()
        self.input_layernorm = RMSNorm(cfg.hidden_size, cfg.rms_eps)
        self.self_attn = Attention(cfg, layer_idx)
        self.post_attention_layernorm = RMSNorm(cfg.hidden_size, cfg.rms_eps)
        self.mlp = MLP(cfg)

    def forward(self, delta, res, rope_table, ctx, parts: bool = False):
        """Carries the residual stream as (delta, res) with hidden =
        delta + res: the pending add fuses into the NEXT norm's kernel
        (ops.add_rms_norm), so no standalone residual-add kernels run.  So does the sum
        of a decoding projection's parts (ops.linear_parts), of this layer's last one
        only if the caller asks for `parts`."""
        eps, few = self.input_layernorm.eps, _few(delta.shape[-2])
        a_in, h = ops.add_parts_rms_norm(delta, res, self.input_layernorm.weight, eps)
        attn_delta = self.self_attn(a_in, rope_table, ctx,
                                    **(_parts(self.self_attn, Attention) if few else {}))
        m_in, h2 = ops.add_parts_rms_norm(attn_delta, h,
                                          self.post_attention_layernorm.weight, eps)
        return self.mlp(m_in, **(_parts(self.mlp, MLP) if parts and few else {})), h2


_FORWARDS = {cls: cls.forward for cls in (Attention, MLP, Block)}


class Transformer(nn.Module):
    """Shared backbone (causal or bidirectional by AttnContext.causal)."""

    def __init__(self, cfg: ModelConfig):
        super().__init__()
        self.cfg = cfg
        self.embed_tokens = nn.Embedding(cfg.vocab_size, cfg.hidden_size)
        self.layers = nn.ModuleList(Block(cfg, i) for i in range(cfg.num_layers))
        self.norm = RMSNorm(cfg.hidden_size, cfg.rms_eps)
        table = ops.build_rope_cache(cfg.head_dim, cfg.max_position, cfg.rope_theta)
        self.register_buffer("rope_table", table, persistent=False)

    def forward(self, input_ids: torch.Tensor, ctx: AttnContext,
                checkpoint: bool = False) -> torch.Tensor:
        if self.rope_table.dtype != torch.float32:
            # keep the rope table fp32 even after model.to(bf16)
            self.rope_table = self.rope_table.float()
        delta = self.embed_tokens(input_ids)
        res = None
        layers, few = list(self.layers), _few(delta.shape[0])
        plain = few and layers and _plain(layers[0], Block)
        for i, layer in enumerate(layers):
            if checkpoint and torch.is_grad_enabled():
                delta, res = torch.utils.checkpoint.checkpoint(
                    layer, delta, res, self.rope_table, ctx, use_reentrant=False)
            else:
                # parts only for a next layer that knows of them, or the norm below
                then = few and (i + 1 == len(layers) or _plain(layers[i + 1], Block))
                delta, res = layer(delta, res, self.rope_table, ctx,
                                   **(dict(parts=True) if plain and then else {}))
                plain = then
        y, _ = ops.add_parts_rms_norm(delta, res, self.norm.weight, self.norm.eps)
        return y


class CausalLM(nn.Module):
    extensions = ("_C", "_serve")       # HIP extensions its forward needs
    kv_cache_dtypes = ("fp8_e4m3", "bf16")
    packed_prefill = True               # whole prompts run without reading the cache

    def __init__(self, cfg: ModelConfig):
        super().__init__()
        self.cfg = cfg
        self.model = Transformer(cfg)
        if cfg.tie_word_embeddings:
            self.lm_head = None
        else:
            self.lm_head = nn.Linear(cfg.hidden_size, cfg.vocab_size, bias=False)
        self.gradient_checkpointing = False
        self.apply(self._init_weights)

    def _init_weights(self, m):
        if isinstance(m, nn.Linear):
            nn.init.normal_(m.weight, std=0.02)
            if m.bias is not None:
                nn.init.zeros_(m.bias)
        elif isinstance(m, nn.Embedding):
            nn.init.normal_(m.weight, std=0.02)

    @property
    def lm_head_weight(self) -> torch.Tensor:
        if self.lm_head is not None:
            return self.lm_head.weight
        return self.model.embed_tokens.weight

    def forward(self, input_ids: torch.Tensor, ctx: AttnContext) -> torch.Tensor:
        """Returns final hidden states [T, H] (logits are computed by the
        caller via ops.token_logprob_entropy or .logits())."""
        return self.model(input_ids, ctx, checkpoint=self.gradient_checkpointing)

    def logits(self, hidden: torch.Tensor) -> torch.Tensor:
        return ops.linear(hidden, self.lm_head_weight)

    @staticmethod
    def train_ctx(cu_seqlens: torch.Tensor, max_seqlen: int, positions: torch.Tensor,
                  causal: bool = True) -> AttnContext:
        return AttnContext(mode="train", positions=positions, cu_seqlens=cu_seqlens,
                           max_seqlen=max_seqlen, causal=causal)

    @classmethod
    def from_preset(cls, name: str, **overrides) -> "CausalLM":
        return cls(get_config(name, **overrides))


def make_positions(cu_seqlens: torch.Tensor) -> torch.Tensor:
    """position ids 0..len-1 per packed sequence (one wait for the device, for the
    boundaries: repeat_interleave would write past its output where they fall)."""
    bounds = cu_seqlens.tolist()
    if any(b < a for a, b in zip(bounds, bounds[1:])):
        raise RuntimeError(f"sequence boundaries must not fall: {bounds}")
    first = cu_seqlens[:-1].long()
    T = bounds[-1] - bounds[0] if len(bounds) > 1 else 0
    starts = torch.repeat_interleave(first - cu_seqlens[0].long() if T else first,
                                     (cu_seqlens[1:] - cu_seqlens[:-1]).long(), output_size=T)
    return torch.arange(T, device=cu_seqlens.device) - starts


def pack_sequences(seqs: list[torch.Tensor], device="cpu"):
    """Pack a list of 1-D id tensors → (input_ids [T], cu_seqlens [B+1] int32,
    max_seqlen, positions [T])."""
    lens = [int(s.numel()) for s in seqs]
    cu = torch.zeros(len(seqs) + 1, dtype=torch.int32, device=device)
    cu[1:] = torch.cumsum(torch.tensor(lens, dtype=torch.int32, device=device), 0)
    ids = torch.cat([s.to(device) for s in seqs]) if seqs else torch.zeros(0, dtype=torch.long)
    pos = make_positions(cu)
    return ids.long(), cu, (max(lens) if lens else 0), pos
