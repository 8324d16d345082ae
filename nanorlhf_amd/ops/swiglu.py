"""Fused SwiGLU activation: y = silu(gate) * up, with gate/up interleaved as
one [N, 2*I] tensor (the gate_up projection's output).  Fusing halves the
HBM round-trips vs separate silu+mul."""
from __future__ import annotations

import torch

from . import ext, linear_ext, serve_ext
from .linear import differentiated, few_rows, here, linear, plain_call


def _swiglu_ref(gate_up: torch.Tensor) -> torch.Tensor:
    gate, up = gate_up.chunk(2, dim=-1)
    return (torch.nn.functional.silu(gate.float()) * up.float()).to(gate_up.dtype)


class _SwigluFn(torch.autograd.Function):
    @staticmethod
    def forward(ctx, gate_up):
        ctx.save_for_backward(gate_up)
        return ext().swiglu_fwd(gate_up)

    @staticmethod
    def backward(ctx, dy):
        (gate_up,) = ctx.saved_tensors
        return ext().swiglu_bwd(dy.contiguous(), gate_up)


def swiglu(gate_up: torch.Tensor) -> torch.Tensor:
    if gate_up.is_cuda and not differentiated(gate_up):
        return ext().swiglu_fwd(gate_up.contiguous())
    if gate_up.is_cuda:
        return _SwigluFn.apply(gate_up.contiguous())
    return _swiglu_ref(gate_up)


# Rows and depths from and up to which both products and the activation are one
# kernel.  Library product and a pass against it, in us: 1024 x 4864 x 896 40 / 25,
# 2048 x 4096 x 1024 68 / 33, 600 x 8960 x 1536 51 / 40, 16320 x 8960 x 1536 857 /
# 786.  A few rows leave most of its 256-row tiles empty (300 x 8960 x 1536: 34 /
# 37), deep products have little to save (4096 x 18944 x 3584: 872 / 910), and its tiles
# have to fill the CUs' rounds (glu_fills).
GLU_ROWS, GLU_DEPTH = 512, 2048
# Fewer rows are about as fast by it, and a library call (19 us of the host's time) and a launch
# less, where 36 tiles of columns or more keep CUs at work and, in the deeper ones, 70 tiles do and
# the last 256 rows are more than half there.  In us, over operands that no cache holds: 212 x 4864
# x 896 17.4 / 17.9, 400 21.1 / 18.9, 192 x 8192 x 896 as the slowest 0.86 of the rate; 212 x 8960
# x 1536 32.9 / 33.2, 385 37.0 / 35.3, 212 x 11008 x 2048 41.6 / 40.4; but 192 x 6144 x 1536, of 48
# tiles, 23.0 / 29.4, 288 x 7168 x 1536 0.95, 257 x 4608 x 1536 0.83, and with the weights in
# caches 128 x 4864 x 896 12.2 / 15.7, 212 x 4096 x 1024 13.5 / 16.8, 328 x 8960 x 1536 28.6 / 31.3.
GLU_FEWER, GLU_WIDE = 192, 36 * 128
# The kernel of few rows does not divide the depth: 16 rows of 4128 x 8192 take the library
# and a pass 36 us, it 45, of 4128 x 4096 28 and 23.
FEW_DEPTH = 4096


def glu_fills(M: int, I: int, K: int) -> bool:
    """Whether M x I x K fills enough of the rounds that 256 CUs need for its tiles of 256 x
    128, one each: a tile's time grows with the depth, an idle CU's share of it with that.
    Library and pass / kernel in us: 512 x 1024 x 1536 13.5 / 31.6 (8 tiles), 1024 x 2240 x
    1536 25.8 / 32 (72), 2000 x 2240 x 1536 43 / 34 (144), 600 x 11008 x 2048 70 / 88 (258);
    512 x 4864 x 896 25 / 21 (76).  A shallow product is launches."""
    tiles = -(-M // 256) * -(-I // 128)
    return K <= 256 or tiles / (256 * -(-tiles // 256)) >= (0.25 if K <= 1024 else 0.6)


def glu_pays(M: int, I: int, K: int) -> bool:
    if M >= GLU_ROWS:
        return glu_fills(M, I, K)
    return M >= GLU_FEWER and I >= GLU_WIDE and (
        K <= 1024 or (M - 1) % 256 >= 128 and -(-M // 256) * -(-I // 128) >= 70)


def glu_fuses(x: torch.Tensor, gate: torch.Tensor) -> bool:
    """Whether glu_linear takes (and is the faster way for) these operands."""
    return (here(x) and plain_call(x, gate) and x.dim() == 2
            and x.dtype == gate.dtype == torch.bfloat16 and x.is_contiguous()
            and gate.is_contiguous() and gate.device == x.device
            and x.shape[1] % 64 == 0 and 0 < x.shape[1] <= GLU_DEPTH
            and x.data_ptr() % 16 == 0 and gate.data_ptr() % 16 == 0
            and glu_pays(x.shape[0], gate.shape[0], x.shape[1]))


def linear_swiglu(x: torch.Tensor, weight: torch.Tensor) -> torch.Tensor:
    """swiglu of x [..., K] times weight [2 I, K] (gate rows, then up rows)."""
    gate, up = weight.chunk(2)
    if few_rows(x, gate) and x.shape[1] <= FEW_DEPTH:
        return linear_ext().glu_rows(x, gate, up)
    if not glu_fuses(x, gate):
        return swiglu(linear(x, weight))
    out = torch.empty(x.shape[0], gate.shape[0], dtype=x.dtype, device=x.device)
    linear_ext().glu_linear(x, gate, up, out, 0)
    return out


def relu_squared_(x: torch.Tensor) -> torch.Tensor:
    """x <- relu(x)^2, in place."""
    if x.is_cuda:
        serve_ext().relu_squared_(x)
        return x
    return x.copy_(torch.relu(x.float()).pow(2))


def linear_gelu_glu(x: torch.Tensor, gate: torch.Tensor, up: torch.Tensor,
                    out: torch.Tensor) -> None:
    """out = gelu_tanh(x gate^T) * (x up^T), where glu_fuses(x, gate); out may be
    columns of a wider row."""
    linear_ext().glu_linear(x, gate, up, out, 1)


def gelu_glu(gate: torch.Tensor, up: torch.Tensor, out: torch.Tensor,
             pad: int = 0, tail: int = 0) -> None:
    """out[:, pad:pad+ff] = gelu_tanh(gate) * up; the pad columns ahead and the
    tail columns behind are zeroed.  gate, up and out are column slices."""
    if gate.is_cuda:
        serve_ext().gelu_glu(gate, up, out, pad, tail)
        return
    ff = gate.shape[1]
    out[:, :pad] = 0
    out[:, pad + ff:] = 0
    g = torch.nn.functional.gelu(gate.float(), approximate="tanh")
    out[:, pad:pad + ff] = (g * up.float()).to(out.dtype)
