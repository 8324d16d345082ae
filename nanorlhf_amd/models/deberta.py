"""DeBERTa-v2/v3 sequence-classification reward model (own implementation).

The reference's reward model is microsoft/deberta-v3-large loaded through
AutoModelForSequenceClassification (GRPO/grpo.py:162-198).
This module implements that architecture —
disentangled attention with log-bucketed relative positions (c2p + p2c,
shared q/k projections for the position embeddings), LayerNorm/GELU
encoder, context pooler + classifier head — and imports real HF
safetensors checkpoints by name.

Correctness is pinned by tests/test_deberta.py: outputs are compared
against transformers' DebertaV2ForSequenceClassification on random
weights (transformers is a local test oracle only — no transformers code
runs in the training path).

Compute notes (MI355X): the RM scores ≤512-token sequences in large
batches; the S×S disentangled bias makes flash-style fusion unprofitable
at this size (K/V L2-resident — cdna_hip_programming.md common-mistake
#7), so the hot path is hipBLASLt GEMMs over padded batches, which
rocprof shows memory/GEMM bound.  fp32 statistics everywhere LayerNorm
needs them.
"""
from __future__ import annotations

import json
import math
import os
from dataclasses import dataclass
from typing import Optional

import torch
import torch.nn as nn
import torch.nn.functional as F


@dataclass
class DebertaConfig:
    vocab_size: int = 128100
    hidden_size: int = 1024
    num_layers: int = 24
    num_heads: int = 16
    intermediate_size: int = 4096
    max_position_embeddings: int = 512
    position_buckets: int = 256
    max_relative_positions: int = -1     # -1 → max_position_embeddings
    layer_norm_eps: float = 1e-7
    position_biased_input: bool = False  # v3-large: no absolute positions
    num_labels: int = 1
    pooler_hidden_act: str = "gelu"

    @property
    def pos_ebd_size(self) -> int:
        if self.position_buckets > 0:
            return self.position_buckets
        return self.rel_span

    @property
    def rel_span(self) -> int:
        return (self.max_relative_positions if self.max_relative_positions > 0
                else self.max_position_embeddings)

    @staticmethod
    def from_hf(path: str, **overrides) -> "DebertaConfig":
        with open(os.path.join(path, "config.json")) as f:
            hf = json.load(f)
        d = dict(
            vocab_size=hf["vocab_size"],
            hidden_size=hf["hidden_size"],
            num_layers=hf["num_hidden_layers"],
            num_heads=hf["num_attention_heads"],
            intermediate_size=hf["intermediate_size"],
            max_position_embeddings=hf.get("max_position_embeddings", 512),
            position_buckets=hf.get("position_buckets", -1),
            max_relative_positions=hf.get("max_relative_positions", -1),
            layer_norm_eps=hf.get("layer_norm_eps", 1e-7),
            position_biased_input=hf.get("position_biased_input", True),
            num_labels=len(hf.get("id2label", {0: None})) or 1,
            pooler_hidden_act=hf.get("pooler_hidden_act", "gelu"),
        )
        d.update(overrides)
        return DebertaConfig(**d)


def make_log_bucket_position(rel: torch.Tensor, bucket: int, max_pos: int) -> torch.Tensor:
    """Log-bucketed relative positions (DeBERTa-v2 scheme): exact within
    ±bucket/2, logarithmic buckets out to max_pos beyond."""
    sign = torch.sign(rel).to(torch.float32)
    mid = bucket // 2
    abs_pos = torch.where((rel < mid) & (rel > -mid),
                          torch.full_like(rel, mid - 1), rel.abs()).float()
    log_pos = torch.ceil(torch.log(abs_pos / mid)
                         / math.log((max_pos - 1) / mid) * (mid - 1)) + mid
    return torch.where(abs_pos <= mid, rel.float(), log_pos * sign).long()


def build_relative_position(q_len: int, k_len: int, bucket: int, max_pos: int,
                            device) -> torch.Tensor:
    rel = (torch.arange(q_len, device=device)[:, None]
           - torch.arange(k_len, device=device)[None, :])
    if bucket > 0 and max_pos > 0:
        rel = make_log_bucket_position(rel, bucket, max_pos)
    return rel  # [q_len, k_len] long


class DisentangledSelfAttention(nn.Module):
    """c2p + p2c disentangled attention, share_att_key=True (v3)."""

    def __init__(self, cfg: DebertaConfig):
        super().__init__()
        self.cfg = cfg
        H = cfg.hidden_size
        self.num_heads = cfg.num_heads
        self.head_dim = H // cfg.num_heads
        self.query_proj = nn.Linear(H, H)
        self.key_proj = nn.Linear(H, H)
        self.value_proj = nn.Linear(H, H)

    def _heads(self, x: torch.Tensor) -> torch.Tensor:
        # [B, S, H] -> [B, h, S, d]
        B, S, _ = x.shape
        return x.view(B, S, self.num_heads, self.head_dim).transpose(1, 2)

    def forward(self, x: torch.Tensor, mask2d: torch.Tensor,
                rel_pos: torch.Tensor, rel_emb: torch.Tensor) -> torch.Tensor:
        cfg = self.cfg
        B, S, H = x.shape
        q = self._heads(self.query_proj(x))
        k = self._heads(self.key_proj(x))
        v = self._heads(self.value_proj(x))
        scale = math.sqrt(self.head_dim * 3)  # 1 + c2p + p2c
        att = (q @ k.transpose(-1, -2)) / scale

        span = cfg.pos_ebd_size
        pe = rel_emb[: span * 2]                            # [2*span, H]
        pos_q = self.query_proj(pe).view(span * 2, self.num_heads,
                                         self.head_dim).transpose(0, 1)
        pos_k = self.key_proj(pe).view(span * 2, self.num_heads,
                                       self.head_dim).transpose(0, 1)
        # content→position: Q · pos_Kᵀ gathered at bucket(rel)
        c2p = q @ pos_k.transpose(-1, -2)                   # [B, h, S, 2*span]
        idx = (rel_pos + span).clamp(0, span * 2 - 1)       # [S, S]
        att = att + torch.gather(
            c2p, -1, idx.expand(B, self.num_heads, S, S)) / scale
        # position→content: K · pos_Qᵀ gathered at bucket(-rel), transposed
        p2c = k @ pos_q.transpose(-1, -2)
        idx_t = (-rel_pos + span).clamp(0, span * 2 - 1)
        att = att + torch.gather(
            p2c, -1, idx_t.expand(B, self.num_heads, S, S)).transpose(-1, -2) / scale

        att = att.masked_fill(~mask2d[:, None], torch.finfo(att.dtype).min)
        probs = att.softmax(-1)
        o = probs @ v                                       # [B, h, S, d]
        return o.transpose(1, 2).reshape(B, S, H)


class DebertaLayer(nn.Module):
    def __init__(self, cfg: DebertaConfig):
        super().__init__()
        H = cfg.hidden_size
        self.self_attn = DisentangledSelfAttention(cfg)
        self.attn_out = nn.Linear(H, H)
        self.attn_norm = nn.LayerNorm(H, eps=cfg.layer_norm_eps)
        self.inter = nn.Linear(H, cfg.intermediate_size)
        self.out = nn.Linear(cfg.intermediate_size, H)
        self.out_norm = nn.LayerNorm(H, eps=cfg.layer_norm_eps)

    def forward(self, x, mask2d, rel_pos, rel_emb):
        a = self.self_attn(x, mask2d, rel_pos, rel_emb)
        x = self.attn_norm(self.attn_out(a) + x)
        h = F.gelu(self.inter(x))
        x = self.out_norm(self.out(h) + x)
        return x


class DebertaV3Reward(nn.Module):
    """DebertaV2ForSequenceClassification-equivalent scorer."""

    def __init__(self, cfg: DebertaConfig):
        super().__init__()
        self.cfg = cfg
        H = cfg.hidden_size
        self.word_embeddings = nn.Embedding(cfg.vocab_size, H)
        self.position_embeddings = (
            nn.Embedding(cfg.max_position_embeddings, H)
            if cfg.position_biased_input else None)
        self.emb_norm = nn.LayerNorm(H, eps=cfg.layer_norm_eps)
        self.layers = nn.ModuleList(DebertaLayer(cfg) for _ in range(cfg.num_layers))
        self.rel_embeddings = nn.Embedding(cfg.pos_ebd_size * 2, H)
        self.rel_norm = nn.LayerNorm(H, eps=cfg.layer_norm_eps)  # norm_rel_ebd
        self.pooler = nn.Linear(H, H)
        self.classifier = nn.Linear(H, max(cfg.num_labels, 1))

    def forward(self, input_ids: torch.Tensor,
                attention_mask: Optional[torch.Tensor] = None) -> torch.Tensor:
        """input_ids [B, S] (padded), attention_mask [B, S] → logits [B, L]."""
        cfg = self.cfg
        B, S = input_ids.shape
        if attention_mask is None:
            attention_mask = torch.ones_like(input_ids)
        x = self.word_embeddings(input_ids)
        if self.position_embeddings is not None:
            pos = torch.arange(S, device=input_ids.device)
            x = x + self.position_embeddings(pos)[None]
        x = self.emb_norm(x)
        x = x * attention_mask[..., None].to(x.dtype)
        mask2d = (attention_mask[:, None, :] * attention_mask[:, :, None]).bool()
        rel_pos = build_relative_position(S, S, cfg.position_buckets,
                                          cfg.rel_span, input_ids.device)
        rel_emb = self.rel_norm(self.rel_embeddings.weight)
        for layer in self.layers:
            x = layer(x, mask2d, rel_pos, rel_emb)
        pooled = torch.tanh(self.pooler(x[:, 0])) if cfg.pooler_hidden_act == "tanh" \
            else F.gelu(self.pooler(x[:, 0]))
        return self.classifier(pooled)

    # ------------------------------------------------------------- HF import
    @staticmethod
    def hf_key_map(cfg: DebertaConfig) -> dict[str, str]:
        m = {
            "deberta.embeddings.word_embeddings.weight": "word_embeddings.weight",
            "deberta.embeddings.LayerNorm.weight": "emb_norm.weight",
            "deberta.embeddings.LayerNorm.bias": "emb_norm.bias",
            "deberta.encoder.rel_embeddings.weight": "rel_embeddings.weight",
            "deberta.encoder.LayerNorm.weight": "rel_norm.weight",
            "deberta.encoder.LayerNorm.bias": "rel_norm.bias",
            "pooler.dense.weight": "pooler.weight",
            "pooler.dense.bias": "pooler.bias",
            "classifier.weight": "classifier.weight",
            "classifier.bias": "classifier.bias",
        }
        if cfg.position_biased_input:
            m["deberta.embeddings.position_embeddings.weight"] = \
                "position_embeddings.weight"
        for i in range(cfg.num_layers):
            hp = f"deberta.encoder.layer.{i}"
            op = f"layers.{i}"
            for proj in ("query_proj", "key_proj", "value_proj"):
                for wb in ("weight", "bias"):
                    m[f"{hp}.attention.self.{proj}.{wb}"] = f"{op}.self_attn.{proj}.{wb}"
            for wb in ("weight", "bias"):
                m[f"{hp}.attention.output.dense.{wb}"] = f"{op}.attn_out.{wb}"
                m[f"{hp}.attention.output.LayerNorm.{wb}"] = f"{op}.attn_norm.{wb}"
                m[f"{hp}.intermediate.dense.{wb}"] = f"{op}.inter.{wb}"
                m[f"{hp}.output.dense.{wb}"] = f"{op}.out.{wb}"
                m[f"{hp}.output.LayerNorm.{wb}"] = f"{op}.out_norm.{wb}"
        return m

    def load_hf_state(self, hf_state: dict[str, torch.Tensor]) -> "DebertaV3Reward":
        key_map = self.hf_key_map(self.cfg)
        own = {}
        for hk, ok in key_map.items():
            if hk not in hf_state:
                raise KeyError(f"DeBERTa checkpoint missing {hk!r}")
            own[ok] = hf_state[hk]
        missing, unexpected = self.load_state_dict(own, strict=False)
        if missing:
            raise RuntimeError(f"unmapped model keys: {missing[:6]}")
        return self

    @classmethod
    def from_pretrained(cls, path: str, **overrides) -> "DebertaV3Reward":
        from .hf_import import load_hf_tensors
        cfg = DebertaConfig.from_hf(path, **overrides)
        model = cls(cfg)
        return model.load_hf_state(load_hf_tensors(path))


class DebertaReward:
    """String-contract reward closure over a DebertaV3Reward + its own
    tokenizer, mirroring the reference reward_func (GRPO/grpo.py:162-198):
    re-tokenizes decoded strings with the RM tokenizer (truncation 512),
    batched forward at reward_batch_size."""

    def __init__(self, model: DebertaV3Reward, tokenizer, device,
                 batch_size: int = 16, max_len: int = 512,
                 offload=None):
        self.model = model
        self.tokenizer = tokenizer
        self.device = torch.device(device)
        self.batch_size = batch_size
        self.max_len = max_len
        self.offload = offload

    @torch.no_grad()
    def __call__(self, texts: list[str]) -> torch.Tensor:
        if self.offload is not None:
            self.offload.model_to_device(self.model)
            self.offload.join_compute()
        self.model.eval()
        scores = []
        for i in range(0, len(texts), self.batch_size):
            batch = texts[i: i + self.batch_size]
            enc = self.tokenizer(batch, padding=True, truncation=True,
                                 max_length=self.max_len, return_tensors="pt")
            logits = self.model(enc["input_ids"].to(self.device),
                                enc["attention_mask"].to(self.device))
            scores.append(logits[:, 0].float().cpu())
        if self.offload is not None and self.offload.should_offload():
            self.offload.model_to_host(self.model)
        return torch.cat(scores)
