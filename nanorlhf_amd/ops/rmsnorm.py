"""RMSNorm forward/backward.

Replaces transformers' Qwen2RMSNorm used inside every reference model call.  GPU path is a fused HIP
kernel (one pass, bf16x8 vector loads, fp32 accumulation)."""
from __future__ import annotations

import torch

from . import ext, serve_ext
from .linear import plain_call, sum_parts


def _rms_norm_ref(x: torch.Tensor, weight: torch.Tensor, eps: float) -> torch.Tensor:
    dtype = x.dtype
    xf = x.float()
    inv = torch.rsqrt(xf.pow(2).mean(-1, keepdim=True) + eps)
    return (xf * inv).to(dtype) * weight


class _RMSNormFn(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, weight, eps):
        y, invrms = ext().rmsnorm_fwd(x, weight, eps)
        ctx.save_for_backward(x, weight, invrms)
        return y

    @staticmethod
    def backward(ctx, dy):
        x, weight, invrms = ctx.saved_tensors
        want_dw = ctx.needs_input_grad[1]      # not for a frozen weight, as under LoRA
        dx, dw = ext().rmsnorm_bwd(dy.contiguous(), x, weight, invrms, want_dw=want_dw)
        return dx, dw if want_dw else None, None


def rms_norm(x: torch.Tensor, weight: torch.Tensor, eps: float = 1e-6) -> torch.Tensor:
    if x.is_cuda:
        return _RMSNormFn.apply(x.contiguous(), weight, eps)
    return _rms_norm_ref(x, weight, eps)


class _AddRMSNormFn(torch.autograd.Function):
    """h = x + res; y = rmsnorm(h)*w — fused (one kernel, h register-resident
    for H<=2048).  Backward: dh = rmsnorm_bwd(dy, h) and the grads of x and
    res are both dh (+ whatever later consumers of h contributed)."""

    @staticmethod
    def forward(ctx, x, res, weight, eps):
        y, h, invrms = ext().rmsnorm_addres_fwd(x, res, weight, eps)
        ctx.save_for_backward(h, weight, invrms)
        return y, h

    @staticmethod
    def backward(ctx, dy, dh_out):
        h, weight, invrms = ctx.saved_tensors
        want_dw = ctx.needs_input_grad[2]
        if dh_out is not None:
            dh_out = dh_out.contiguous()
        recorded = torch.is_grad_enabled() and dh_out is not None    # a second derivative
        dh, dw = ext().rmsnorm_bwd(dy.contiguous(), h, weight, invrms,
                                   None if recorded else dh_out, want_dw)
        if recorded:
            dh = dh + dh_out
        return dh, dh, dw if want_dw else None, None


def add_rms_norm(x: torch.Tensor, res: torch.Tensor | None, weight: torch.Tensor,
                 eps: float = 1e-6):
    """Fused residual-add + RMSNorm: returns (normed, h=x+res).  res=None →
    plain rms_norm (h = x)."""
    if res is None:
        return rms_norm(x, weight, eps), x
    if x.is_cuda and x.dtype == torch.bfloat16:
        return _AddRMSNormFn.apply(x.contiguous(), res.contiguous(), weight, eps)
    h = x + res
    return rms_norm(h, weight, eps), h


def add_parts_rms_norm(x: torch.Tensor, res: torch.Tensor | None, weight: torch.Tensor,
                       eps: float = 1e-6):
    """add_rms_norm, of linear_parts' result."""
    if x.dim() != 3 or x.dtype != torch.float32 or res is None or res.dim() != 2:
        return add_rms_norm(x, res, weight, eps)
    if x.is_cuda and plain_call(x, res, weight) and x.shape[0] <= 8 and x.shape[2] % 8 == 0 \
            and res.dtype == weight.dtype == torch.bfloat16 \
            and weight.device == res.device == x.device and weight.is_contiguous() \
            and all(t.is_contiguous() and t.data_ptr() % 16 == 0 for t in (x, res, weight)):
        return tuple(ext().rmsnorm_parts_fwd(x, res, weight, eps))
    return add_rms_norm(sum_parts(x, res.dtype), res, weight, eps)


def _group_rms(x: torch.Tensor, groups: int, eps: float) -> torch.Tensor:
    parts = x.float().unflatten(-1, (groups, x.shape[-1] // groups))
    parts = parts * torch.rsqrt(parts.pow(2).mean(-1, keepdim=True) + eps)
    return parts.flatten(-2)


def residual_group_norm(x: torch.Tensor, weight: torch.Tensor | None, eps: float, *,
                        groups: int = 1, delta: torch.Tensor | None = None,
                        mult: float = 1.0, embed: torch.Tensor | None = None,
                        ids: torch.Tensor | None = None, add: torch.Tensor | None = None,
                        bias: torch.Tensor | None = None, offset: float = 0.0,
                        gain: float = 1.0) -> torch.Tensor:
    """Norm of a 32-bit residual stream, with the pending update fused in.

    x [T, W] float32 is changed IN PLACE: set to embed[ids] if `ids` is given,
    else x += mult * delta if `delta` is.  delta may be [T, parts, W], whose
    parts are all added.  add [T, W] float32 and bias [W] are added to x too.
    Returns, in the weight's dtype, x split into `groups` equal
    parts, each divided by its own root mean square, times (offset + weight
    [W]) * gain; without a weight, x itself in delta's dtype."""
    if x.is_cuda:
        return serve_ext().residual_group_norm(x, delta, embed, ids, add, bias, weight, groups,
                                               float(mult), float(eps), float(offset),
                                               float(gain))
    if ids is not None:
        x.copy_(embed[ids])
    if add is not None:
        x.add_(add)
    if bias is not None:
        x.add_(bias.float())
    if delta is not None:
        x.add_((delta.float() if delta.dim() == 2 else delta.float().sum(1)) * mult)
    if weight is None:
        return x.to(delta.dtype)
    return (_group_rms(x, groups, eps) * (offset + weight.float()) * gain).to(weight.dtype)


def gated_norm(x: torch.Tensor, weight: torch.Tensor | None, gate: torch.Tensor,
               out: torch.Tensor, eps: float, *, groups: int = 1,
               act: str = "silu") -> None:
    """out[:] = grouped RMS norm of x (times weight) times act(gate); act is
    "silu" or "sigmoid".  gate and out are column slices of wider rows."""
    if x.is_cuda:
        serve_ext().gated_norm(x, weight, gate, out, groups,
                               {"silu": 0, "sigmoid": 1}[act], float(eps))
        return
    y = _group_rms(x, groups, eps)
    if weight is not None:
        y = y * weight.float()
    g = gate.float()
    out.copy_(y * (g * torch.sigmoid(g) if act == "silu" else torch.sigmoid(g)))
