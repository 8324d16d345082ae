"""Linears without gradients.  Few rows (decoding) take csrc/linear_rows.hip, which
is bound by reading the weights; the rest is the library's."""
from __future__ import annotations

import torch
import torch.autograd.forward_ad as forward_ad
import torch.nn.functional as F
from torch.utils._device import DeviceContext

from . import linear_ext

# Library against the kernel, in us: 64 rows of 3584 x 18944 91 / 36, of 4608 x 3584
# 18.7 / 15.3, of 151936 x 1536 115 / 108; with more rows x weighs as much as the weights
# and the library's tiles share it better.
FEW_ROWS = 64
DEPTH = 1 << 24         # from which on its 32-bit offsets would wrap


def unwatched(*tensors: torch.Tensor) -> bool:
    """Whether nobody traces, transforms or listens to calls on these: no forward-mode
    derivative, no trace or transform, no mode of dispatch or of functions (but the one
    that only gives new tensors their device), no tensor that overrides its calls."""
    return not (forward_ad._current_level >= 0 or torch.jit.is_tracing()
                or torch.compiler.is_compiling()
                or torch._C._functorch.peek_interpreter_stack() is not None
                or torch._C._len_torch_dispatch_stack()
                or torch._ops._len_torch_dispatch_stack_pre_dispatch()
                or any(type(torch._C._get_function_stack_at(i)) is not DeviceContext
                       for i in range(torch._C._len_torch_function_stack()))) \
        and all(type(t) in (torch.Tensor, torch.nn.Parameter) for t in tensors)


def plain_call(*tensors: torch.Tensor) -> bool:
    """Whether a library call on these may be replaced by a kernel: no gradient, no
    autocast, and unwatched."""
    return not (torch.is_grad_enabled() or torch.is_autocast_enabled()) and unwatched(*tensors)


def here(x: torch.Tensor) -> bool:
    """Whether x is on the current GPU, on whose stream the kernels are launched; a
    library call goes to its operands' GPU, whichever is the current."""
    return x.is_cuda and x.device.index == torch.cuda.current_device()


def rows_pay(M: int, N: int, K: int) -> bool:
    """Whether M <= FEW_ROWS rows of N x K are faster by the kernel.  Wide products are a
    matter of how full the CUs' last round of 64 columns each is, and from some rows on of
    x's fetch into every CU, which the library's tiles share; deep ones of a few columns
    are divided, deep and wide ones are not.  Library / kernel in us: 32 rows of 18944 x
    1536 16.8 / 19.3, of 32768 x 1536 24.1 / 23.5; 48 rows of 24576 x 1536 20 / 22, of
    16384 x 1536 19.2 / 15; 64 rows of 12288 x 1536 13.6 / 15.3, of 12288 x 896 12 / 10.6;
    16 rows of 14336 x 4096 31 / 25, 32 rows 27 / 30; 1 row of 6144 x 8192 24 / 30."""
    if K > 2048 and N > 5120:
        return M <= 16 and K <= 4096
    tiles = -(-N // 64)
    full = tiles / (256 * -(-tiles // 256)) >= 0.8
    return N <= 16384 or N > 65536 or M <= (32 if full else 16)


def few_rows(x: torch.Tensor, w: torch.Tensor) -> bool:
    """Whether the kernels for few rows can take x [M, K] and w [N, K]."""
    return (here(x) and x.dim() == 2 and x.shape[0] <= FEW_ROWS and plain_call(x, w)
            and x.dtype == w.dtype == torch.bfloat16 and x.shape[1] % 64 == 0
            and x.shape[1] < DEPTH and x.is_contiguous() and w.is_contiguous()
            and w.device == x.device and x.data_ptr() % 16 == 0 and w.data_ptr() % 16 == 0)


def _rows(x: torch.Tensor, w: torch.Tensor, bias: torch.Tensor | None) -> bool:
    return few_rows(x, w) and rows_pay(x.shape[0], *w.shape) and (
        bias is None or plain_call(bias) and bias.dtype == x.dtype
        and bias.device == x.device and bias.shape == w.shape[:1] and bias.is_contiguous())


def linear(x: torch.Tensor, w: torch.Tensor, bias: torch.Tensor | None = None) -> torch.Tensor:
    """x w^T + bias."""
    if _rows(x, w, bias):
        return linear_ext().linear_rows(x, w, bias)
    return F.linear(x, w, bias)


def linear_parts(x: torch.Tensor, w: torch.Tensor, bias: torch.Tensor | None = None):
    """x w^T + bias for a kernel that can add up parts as it reads them: [M, N], or, where
    the depth is divided among workgroups, float32 parts [parts, M, N] of x w^T without the
    bias.  See sum_parts for what they stand for."""
    if _rows(x, w, bias):
        return linear_ext().linear_rows_parts(x, w, bias)
    return F.linear(x, w, bias)


def sum_parts(y: torch.Tensor, dtype: torch.dtype,
              bias: torch.Tensor | None = None) -> torch.Tensor:
    """What linear_parts' result stands for."""
    if y.dim() == 2:
        return y
    s = y[0]
    for p in y[1:]:
        s = s + p
    return (s if bias is None else s + bias.float()).to(dtype)
