"""Sequence mixers: those of the parallel-block models, and (at the end) those
of the sequential-block models.

A parallel block's mixer owns no GEMM: its block projects the normed input once for all of the
mixer's inputs and the feed-forward's, hands it the columns, and gives it
columns of the row that the block's one output GEMM reads.  A mixer says

    inputs       name -> width of the projections it reads
    out_width    width of what it writes
    cache_spec   what it keeps of a sequence (KVSpec or StateSpec)
    weights      its own small parameters: tensor name -> parameter

and computes forward(cols, proj, ctx, cache, out), where cols[name] is the
(first, last) column of an input in proj [T, ld].
"""
from __future__ import annotations

import torch
import torch.nn as nn
import torch.nn.functional as F

from .. import ops
from .config import KVSpec, LatentSpec, StateSpec
from .lora import project


class LinearMixer(nn.Module):
    """Decayed linear attention: the two mixers below differ in what happens to
    q, k, v on the way in and to the output on the way out."""

    silu_inputs = False

    def __init__(self, m: dict, eps: float):
        super().__init__()
        self.heads, self.dim, self.vdim = m["heads"], m["dim"], m["vdim"]
        if len(m["decay"]) != self.heads:
            raise ValueError("one decay per head expected")
        self.decay = ops.DecayTable(m["decay"])
        self.eps = eps
        self.rotation = None
        self.kscale = 1.0
        qk, v = self.heads * self.dim, self.heads * self.vdim
        self.inputs = {"q": qk, "k": qk, "v": v, "g": v}
        self.out_width = v
        self.cache_spec = StateSpec(self.heads, self.dim, self.vdim)

    @property
    def weights(self) -> dict:
        return {}

    def _kw(self, ctx, a, b):
        kw = dict(silu=self.silu_inputs, kscale=self.kscale)
        if self.rotation is not None and self.rotation.dims:
            kw.update(cs=ctx.angles(self.rotation)[a:b], interleaved=self.rotation.interleaved)
        return kw

    def forward(self, cols, proj, ctx, state, out):
        q, k, v, g = (proj[:, cols[n][0]:cols[n][1]] for n in ("q", "k", "v", "g"))
        T, nd = proj.shape[0], ctx.n_decode
        if nd:
            kw = self._kw(ctx, 0, nd)
            self.run(lambda **f: ops.linear_attn_decode(
                q[:nd], k[:nd], v[:nd], self.decay, ctx.state_slots, ctx.seq_lens, state,
                **kw, **f), g[:nd], out[:nd])
        if ctx.portions is not None:
            kw = self._kw(ctx, nd, T)
            self.run(lambda **f: ops.linear_attn_chunked(
                q[nd:], k[nd:], v[nd:], self.decay, ctx.portions, state, **kw, **f),
                g[nd:], out[nd:])


class Retention(LinearMixer):
    """Rotated q and k, k / sqrt(dim); each head's output is divided by its
    root mean square and gated by silu."""

    def __init__(self, m: dict, eps: float):
        super().__init__(m, eps)
        self.rotation = ops.Rotation(m["rot"]["dims"], m["rot"]["base"])
        self.kscale = self.dim ** -0.5

    def run(self, attn, g, out):
        attn(gate=g, eps=self.eps, out=out)


class Lightning(LinearMixer):
    """SiLU on q, k and v; the heads' outputs are normed together, with a
    weight, and gated by a sigmoid."""

    silu_inputs = True

    def __init__(self, m: dict, eps: float):
        super().__init__(m, eps)
        self.norm = nn.Parameter(torch.ones(self.out_width))

    @property
    def weights(self):
        return {"norm": self.norm}

    def run(self, attn, g, out):
        ops.gated_norm(attn(), self.norm, g, out, self.eps, act="sigmoid")


class WindowAttention(nn.Module):
    """Softmax attention over a sliding window and the kept first tokens, with
    per-head query/key norms and rotated values."""

    def __init__(self, m: dict, eps: float):
        super().__init__()
        self.heads, self.kv_heads = m["heads"], m["kv_heads"]
        if self.heads % self.kv_heads:
            raise ValueError("query heads must be a multiple of key/value heads")
        self.dim, self.vdim, self.eps = m["dim"], m["vdim"], eps
        self.scale = m["scale"]
        self.size, self.keep = m["mask"]["size"], m["mask"]["keep_first"]
        rot = m["rot"]
        self.rotation = ops.Rotation(rot["dims"], rot["base"], interleaved=True)
        self.v_rotation = ops.Rotation(self.vdim, rot["base"], interleaved=True)
        self.q_norm = nn.Parameter(torch.ones(self.dim))
        self.k_norm = nn.Parameter(torch.ones(self.dim))
        self.inputs = {"q": self.heads * self.dim, "k": self.kv_heads * self.dim,
                       "v": self.kv_heads * self.vdim}
        self.out_width = self.heads * self.vdim
        self.cache_spec = KVSpec(self.kv_heads, ops.pad_head_dim(self.dim),
                                 ops.pad_head_dim(self.vdim))

    @property
    def weights(self):
        return {"q.norm": self.q_norm, "k.norm": self.k_norm}

    def forward(self, cols, proj, ctx, cache, out):
        k_cache, v_cache = cache
        cs_v = ctx.angles(self.v_rotation)
        q = ops.rotary_qkv(proj, tuple(cols[n][0] for n in ("q", "k", "v")), self.heads,
                           self.kv_heads, self.dim, self.vdim, ctx.slots, k_cache, v_cache,
                           q_norm=self.q_norm, k_norm=self.k_norm,
                           cs_qk=ctx.angles(self.rotation) if self.rotation.dims else None,
                           cs_v=cs_v, interleaved=True, eps=self.eps)
        ops.paged_attn(q, k_cache, v_cache, ctx, out, self.scale, size=self.size,
                       keep=self.keep, uncs=cs_v)


MIXERS = {"retention": Retention, "attention": WindowAttention, "lightning": Lightning}


# ------------------------------------------------------- sequential blocks
# The mixers of the sequential-block models are whole sublayers: they own their
# projections and compute forward(h, ctx, cache) -> the residual's update.

class WKV(nn.Module):
    """RWKV-style time mixing: r, k, v, gate and decay each read their own mix
    of the token's input and its predecessor's."""

    def __init__(self, width: int, m: dict, eps: float):
        super().__init__()
        self.heads, self.dim, self.width, self.eps = m["heads"], m["dim"], width, eps
        self.rank = m["decay_rank"]
        n, rank = self.heads * self.dim, -(-self.rank // 32) * 32
        self.mu = nn.Parameter(torch.empty(5, width))          # r, k, v, g, w
        self.proj = nn.Parameter(torch.empty(4, n, width))     # r, k, v, g
        self.w1 = nn.Parameter(torch.empty(rank, width))
        self.w2 = nn.Parameter(torch.empty(n, rank))
        self.w0 = nn.Parameter(torch.empty(n))
        self.u = nn.Parameter(torch.empty(self.heads, self.dim))
        self.norm = nn.Parameter(torch.empty(n))
        self.o = nn.Linear(n, width, bias=False)
        self.cache_spec = StateSpec(self.heads, self.dim, self.dim, shift=width)

    def load(self, take) -> None:
        n, W, rank = self.heads * self.dim, self.width, self.rank
        for i, s in enumerate("rkvgw"):
            self.mu[i].copy_(take("mu." + s, (W,)))
        for i, s in enumerate("rkvg"):
            self.proj[i].copy_(take(s, (n, W)))
        self.w1.zero_()
        self.w2.zero_()
        self.w1[:rank].copy_(take("w1", (rank, W)))
        self.w2[:, :rank].copy_(take("w2", (n, rank)))
        self.w0.copy_(take("w0", (n,)))
        self.u.copy_(take("u", (self.heads, self.dim)))
        self.norm.copy_(take("norm", (n,)))
        self.o.weight.copy_(take("o", (W, n)))

    def forward(self, h, ctx, cache):
        state, last = cache
        mixed = ops.token_shift(h, self.mu, ctx, last)
        r, k, v, g = ops.stacked_linear(mixed[:4], self.proj)
        w = ops.wkv_decay(F.linear(mixed[4], self.w1), self.w2, self.w0)
        return project(self.o, ops.wkv(r, k, v, w, self.u, ctx, state, g, self.norm, self.eps))


class LatentAttention(nn.Module):
    """Causal softmax attention without positions, whose keys and values are
    made from one cached latent vector per token."""

    def __init__(self, width: int, m: dict, eps: float):
        super().__init__()
        self.heads, self.dim, self.vdim = m["heads"], m["dim"], m["vdim"]
        self.rank, self.scale, self.width, self.eps = m["kv_rank"], m["scale"], width, eps
        H, RP = self.heads, ops.pad_latent(self.rank)
        DK, DV = ops.pad_head_dim(self.dim), ops.pad_head_dim(self.vdim)
        self.q_cols = H * DK
        # one projection: the queries (padded per head), then the latent
        self.in_proj = nn.Linear(width, self.q_cols + -(-self.rank // 8) * 8, bias=False)
        self.dkv_norm = nn.Parameter(torch.empty(self.rank))
        self.uk = nn.Parameter(torch.empty(H, DK, RP))
        self.uk_t = nn.Parameter(torch.empty(H, RP, DK))
        self.uv = nn.Parameter(torch.empty(H, DV, RP))
        self.o = nn.Linear(H * self.vdim, width, bias=False)
        self.cache_spec = LatentSpec(RP)

    def load(self, take) -> None:
        H, D, V, R, W = self.heads, self.dim, self.vdim, self.rank, self.width
        for p in (self.in_proj.weight, self.uk, self.uv):
            p.zero_()
        q = self.in_proj.weight[:self.q_cols].unflatten(0, (H, -1))
        q[:, :D].copy_(take("q", (H * D, W)).unflatten(0, (H, D)))
        self.in_proj.weight[self.q_cols:self.q_cols + R].copy_(take("dkv", (R, W)))
        self.dkv_norm.copy_(take("dkv.norm", (R,)))
        self.uk[:, :D, :R].copy_(take("uk", (H * D, R)).unflatten(0, (H, D)))
        self.uv[:, :V, :R].copy_(take("uv", (H * V, R)).unflatten(0, (H, V)))
        self.uk_t.copy_(self.uk.transpose(1, 2))
        self.o.weight.copy_(take("o", (W, H * V)))

    def forward(self, h, ctx, cache):
        proj = project(self.in_proj, h)
        ops.latent_append(proj[:, self.q_cols:self.q_cols + self.rank], self.dkv_norm, self.eps,
                          ctx.slots, cache)
        out = torch.empty(h.shape[0], self.heads * self.vdim, dtype=h.dtype, device=h.device)
        ops.latent_attn(proj[:, :self.q_cols], cache, ctx, self.uk, self.uk_t, self.uv, out,
                        self.scale)
        return project(self.o, out)


SUBLAYER_MIXERS = {"wkv": WKV, "latent_attention": LatentAttention}
