"""Rotary position embedding (NeoX rotate-half layout, Qwen2 semantics).

cos/sin tables are precomputed on host once per model (fp32, [max_pos, D/2])
— on-device trig would turn this memory-bound op VALU-bound.  The HIP kernel applies RoPE in place
to q and k with a sign flag so backward reuses the same kernel with sin
negated (rotation transpose)."""
from __future__ import annotations

import torch

from . import ext, linear_ext, serve_ext
from .linear import differentiated, linear_by, linear_kernel, unwatched


def build_rope_cache(head_dim: int, max_pos: int, theta: float = 1e6,
                     device=None) -> torch.Tensor:
    """Returns [max_pos, head_dim] fp32 table: first half cos, second half sin.
    Computed on the host; device None is torch's default device, where a model
    under construction has its other tensors."""
    half = torch.arange(0, head_dim, 2, dtype=torch.float64, device="cpu")
    inv_freq = 1.0 / (theta ** (half / head_dim))
    t = torch.arange(max_pos, dtype=torch.float64, device="cpu")
    freqs = torch.outer(t, inv_freq)  # [max_pos, D/2]
    table = torch.cat([freqs.cos(), freqs.sin()], dim=-1).float()
    return table.to(torch.get_default_device() if device is None else device)


def _rope_ref(x: torch.Tensor, table: torch.Tensor, positions: torch.Tensor,
              sign: float = 1.0) -> torch.Tensor:
    # x: [T, H, D]; positions: [T]
    D = x.shape[-1]
    cs = table[positions]  # [T, D]
    cos = cs[:, : D // 2].unsqueeze(1)  # [T, 1, D/2]
    sin = cs[:, D // 2:].unsqueeze(1) * sign
    x1 = x[..., : D // 2].float()
    x2 = x[..., D // 2:].float()
    o1 = x1 * cos - x2 * sin
    o2 = x2 * cos + x1 * sin
    return torch.cat([o1, o2], dim=-1).to(x.dtype)


class _RopeFn(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, table, positions):
        ctx.save_for_backward(table, positions)
        return ext().rope_fwd(x.contiguous(), table, positions, 1.0)

    @staticmethod
    def backward(ctx, dy):
        table, positions = ctx.saved_tensors
        dx = ext().rope_fwd(dy.contiguous(), table, positions, -1.0)
        return dx, None, None


def rope_apply(x: torch.Tensor, table: torch.Tensor, positions: torch.Tensor) -> torch.Tensor:
    """x: [T, H, D] (packed tokens), positions: [T] int32/int64."""
    if x.is_cuda:
        return _RopeFn.apply(x, table, positions)
    if x.requires_grad:
        # autograd-composable CPU path
        return _rope_ref(x, table, positions)
    return _rope_ref(x, table, positions)


class _QkvRopeFn(torch.autograd.Function):
    @staticmethod
    def forward(ctx, qkv, table, positions, heads, kv_heads):
        ctx.save_for_backward(table, positions)
        ctx.heads = heads, kv_heads
        return tuple(ext().qkv_rope_fwd(qkv, table, positions, heads, kv_heads))

    @staticmethod
    def backward(ctx, *grads):
        table, positions = ctx.saved_tensors
        grads = [None if g is None else g.contiguous() for g in grads]
        return ext().qkv_rope_bwd(*grads, table, positions, *ctx.heads), None, None, None, None


def split_qkv(qkv: torch.Tensor, heads: int, kv_heads: int):
    """q [T, heads, D], k and v [T, kv_heads, D] of a joint projection's rows."""
    n = heads + 2 * kv_heads
    parts = qkv.unflatten(1, (n, qkv.shape[1] // n))
    return parts.split([heads, kv_heads, kv_heads], dim=1)


def qkv_rope(qkv: torch.Tensor, table: torch.Tensor, positions: torch.Tensor, heads: int,
             kv_heads: int):
    """qkv [T, (heads + 2 kv_heads) D], the heads of q, then k's, then v's: split,
    with q and k rotated as by rope_apply."""
    if qkv.is_cuda and qkv.shape[1] // (heads + 2 * kv_heads) % 16 == 0:
        if not differentiated(qkv):
            return tuple(ext().qkv_rope_fwd(qkv.contiguous(), table, positions, heads, kv_heads))
        return _QkvRopeFn.apply(qkv.contiguous(), table, positions, heads, kv_heads)
    q, k, v = split_qkv(qkv, heads, kv_heads)
    return (rope_apply(q, table, positions), rope_apply(k, table, positions), v)


def linear_qkv_rope(x: torch.Tensor, w: torch.Tensor, bias: torch.Tensor | None,
                    table: torch.Tensor, positions: torch.Tensor, heads: int, kv_heads: int):
    """qkv_rope of linear(x, w, bias), in one kernel where that product is linear_big's."""
    name = linear_kernel(x, w, bias)
    if name == "linear_big" and w.shape[0] in [(heads + 2 * kv_heads) * d for d in (64, 128)] \
            and unwatched(table, positions) \
            and table.dim() == 2 and table.shape[1] * (heads + 2 * kv_heads) == w.shape[0] \
            and table.dtype == torch.float32 and table.is_contiguous() \
            and table.data_ptr() % 8 == 0 and table.device == positions.device == x.device \
            and positions.dtype == torch.int64 and positions.is_contiguous() \
            and positions.numel() == x.shape[0] < 1 << 28:
        return tuple(linear_ext().linear_big_rope(x, w, bias, table, positions, heads, kv_heads))
    return qkv_rope(linear_by(name, x, w, bias), table, positions, heads, kv_heads)


class Rotation:
    """Rotary positions over the first `dims` dimensions, in either layout of
    pairs: rotate-half (i with i + dims/2) or interleaved (2i with 2i + 1).

    No table and no maximum position: the cos | sin rows of the tokens of one
    forward are computed once (64-bit angle, 32-bit result) and shared by all
    layers with the same base and dims."""

    def __init__(self, dims: int, base: float, interleaved: bool = False):
        if dims % 2:
            raise ValueError(f"rotary dims must be even, got {dims}")
        self.dims, self.base, self.interleaved = dims, float(base), interleaved
        self.key = (dims, float(base))
        i = torch.arange(dims // 2, dtype=torch.float64, device="cpu")
        self._freqs = {"cpu": self.base ** (-2.0 * i / max(dims, 1))}

    def freqs(self, device) -> torch.Tensor:
        key = str(device)
        if key not in self._freqs:
            self._freqs[key] = self._freqs["cpu"].to(device)
        return self._freqs[key]

    def angles(self, positions: torch.Tensor) -> torch.Tensor:
        """[T, dims] float32: cos of the dims/2 angles, then sin."""
        f = self.freqs(positions.device)
        if positions.is_cuda:
            return serve_ext().rope_angles(positions, f)
        a = positions.double().unsqueeze(1) * f
        return torch.cat([a.cos(), a.sin()], dim=1).float()


def rotate_pairs(x: torch.Tensor, cs: torch.Tensor, interleaved: bool,
                 sign: float = 1.0) -> torch.Tensor:
    """CPU reference: x [T, H, D] float32, cs [T, dims] with dims <= D."""
    dims = cs.shape[1]
    half = dims // 2
    c = cs[:, None, :half]
    s = cs[:, None, half:] * sign
    if interleaved:
        u, v = x[..., 0:dims:2], x[..., 1:dims:2]
        rot = torch.stack([u * c - v * s, v * c + u * s], dim=-1).flatten(-2)
    else:
        u, v = x[..., :half], x[..., half:dims]
        rot = torch.cat([u * c - v * s, v * c + u * s], dim=-1)
    return torch.cat([rot, x[..., dims:]], dim=-1)
