"""Linears without gradients.  Few rows (decoding) take csrc/linear_rows.hip, which
is bound by reading the weights, and so do more in blocks of 64 while one round of the CUs
takes them all; some thousand take csrc/linear_mid.hip's tiles and many csrc/gemm_big.h's where
those are the faster way, and the rest is the library's."""
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


def differentiated(*tensors: torch.Tensor) -> bool:
    """Whether an autograd function of these has anything to do: a gradient, a forward-mode
    derivative, a transform, or a trace, which records the function to run it again, but of a
    kernel's call only the memory that its result got."""
    if torch.is_grad_enabled():
        for t in tensors:
            if t.requires_grad:
                return True
    return (forward_ad._current_level >= 0 or torch.jit.is_tracing()
            or torch.compiler.is_compiling()
            or torch._C._functorch.peek_interpreter_stack() is not None)


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


BLOCK_ROWS = 1152


def one_round_of_blocks(M: int, N: int) -> bool:
    """Whether M rows and N columns are at most one round of 256 CUs in blocks of 64 x 64."""
    return -(-M // 64) * -(-N // 64) <= 256


def blocks_fill(M: int, N: int) -> bool:
    """Of plain products; many rows of a few columns are the library's (4000 of 64 x 1536 7 us,
    in blocks 10)."""
    return M <= BLOCK_ROWS and one_round_of_blocks(M, N)


def blocks_pay(M: int, N: int, K: int) -> bool:
    """Whether M > FEW_ROWS rows are faster in blocks.  A library call is 19 to 22 us of the
    host's time, the kernel's 5 to 9, which is what counts while a layer's kernels take less;
    on the GPU, library / kernel in us: 130 rows of 2048 x 1536 7.5 / 6.1, 500 9.0 / 8.7; 212
    of 1024 x 1024 5.5 / 4.4, 896 7.8 / 7.3; 896 of 1152 x 896 7.4 / 7.3; 212 of 1536 x 8960
    25.1 / 20.6, 500 28.5 / 28.1; 66 of 3584 x 18944 69 / 39.  Workgroups that leave CUs idle
    over a deep product are not divided, as the library's are: 130 of 1536 x 8960 17.7 / 20.0
    (144 workgroups), 66 of 896 x 4864 8.3 / 8.9 (112).  With two rounds the library's larger
    tiles win: 750 of 1536 x 1536 11.2 / 15.2."""
    if not blocks_fill(M, N):
        return False
    blocks = -(-M // 64)
    groups = next((g for g in (blocks * -(-N // c) for c in (16, 32, 64)) if g <= 256), 256)
    return K <= 4096 or groups >= 154


def mid_fills(M: int, N: int, least: float) -> bool:
    """Whether M rows and N columns are at most one round of 256 CUs in tiles of 128 x 128, and
    at least that part of one."""
    return 256 * least <= -(-M // 128) * -(-N // 128) <= 256


def mid_pays(M: int, N: int, K: int) -> bool:
    """Whether csrc/linear_mid.hip's tiles of 128 x 128 are the faster way for some thousand rows.
    Library / kernel in us: 2667 rows of 1152 x 896 13.2 / 11.5, 1000 of 3072 x 1024 14.2 /
    12.4, 1500 of 2048 x 1536 15.3 / 15.8, 2667 of 1536 x 1536 18.0 / 17.8, with some 14 us less
    of the host's time; half a round or less 1500 of 1152 x 896 9.3 / 10.9, deeper 2667 of
    896 x 4864 35.7 / 35.3, more than a round 4000 of 1152 x 896 13.8 / 20.8.  Few rows of many
    columns and many rows of few, whose tiles are in part empty, over operands that no cache
    holds: up to a depth of 1024 17 to 64 rows of 18944 x 896 15.0 to 13.6 / 11.2 to 12.3, 128 of
    32768 x 1024 20.2 / 18.3, 30000 of 64 x 896 16.5 / 15.3; up to 1536 33 rows of 18944 19.3 / 19.9,
    but 65 25.2 / 22.0, 30000 of 128 26.1 / 28.9, but 9000 of 256 23.6 / 20.7; up to 2048 129 of 8960
    17.8 / 22.0, 128 of 16384 22.5 / 25.9, but 192 of 8960 25.1 / 22.0 (320 of 6144 17.8 / 21.4, as
    the only one of those)."""
    if not mid_fills(M, N, 0.5) or K > 2048:
        return False
    return K <= 1024 or N > 128 and M > (FEW_ROWS if K <= 1536 else 160)


def big_rows(M: int, N: int, K: int) -> bool:
    """Whether M rows are worth tiles of 256: up to three rows of tiles whose last one is more
    than half there, or a few rows of so many columns that they are nearly a round.  Library /
    kernel in us, over operands that no cache holds: 160 rows of 151936 x 1536 141 / 120, 65 122 /
    110, 65 of 65536 54 / 47, 130 of 49152 49 / 44, but of 32768 x 1024 21.4 / 27.1; 257 rows of
    128100 x 1536 152 / 165, 340 of 16640 x 1024 20.6 / 24.0, 513 of 24576 x 1536 54 / 61, but 385 of
    128100 233 / 186, 385 of 16640 23.2 / 24.2, 700 of 18944 x 1024 30.5 / 28.4; 770 of 32768 x 1536
    86 / 75, of 24576 63 / 68."""
    tiles = -(-M // 256) * -(-N // 256)
    if M <= FEW_ROWS:
        return K <= 1024 and tiles >= 256
    return M > 768 or (tiles >= 192 if M <= 256 else (M - 1) % 256 >= 128)


def big_pays(M: int, N: int, K: int) -> bool:
    """Whether csrc/gemm_big.h's tiles of 256 x 256 are the faster way for many rows, by rounds
    of the 256 CUs.  Library / kernel, geometric means over some 20 numbers of rows (lowest,
    highest): from 0.45 rounds on 1.33 (0.99, 1.88) for 1152 x 896, 1.27 for 896 x 896, 1.03
    for 3072 x 1024; with fewer rounds its few tiles' latencies count: 2500 of 1152 x 896 10.6 /
    14.6 us.  Columns that are 256 or a few times as many fit the library's own tiles: 1024 x 896
    and x 1024 0.97 (0.88, 1.33) and 0.92 (0.88, 1.00), 512 x 896 0.91 (0.87, 0.96), but 640 1.26
    (0.99, 1.59), 1280 1.07 (0.91, 1.45); up to 128 columns leave half of each tile empty: 46673
    of 64 x 896 22.3 / 27.2.  From one round on 1.05 (0.95, 1.23) for 2048 x 1536,
    1.04 for 1536 x 1536, 1.03 for 6144 x 1536 and 8960 x 1536.  Up to a depth of 9000 the library
    divides what is no whole round (1536 x 8960 0.98); deeper its choice falls at random on a
    kernel of half its rate: beyond one round and up to five 1.14 (0.85, 1.59) for 1536 x 10496,
    1.16 for 2048 x 13056, 1.20 for 3584 x 18944; 19235 rows of 1536 x 10496 729 / 489 us.  It does
    so below 10240 too, where the library is left what it had: over seven numbers of
    rows of 1536 and 2048 columns 8960 1.08 (0.92, 1.54), 9728 1.09 (0.88, 1.50), 10240 1.11 (0.88,
    1.57), 12288 1.18 (0.96, 1.57)."""
    tiles = -(-M // 256) * -(-N // 256)
    if not big_rows(M, N, K):
        return False
    if K > 2048:
        return K >= 10240 and 256 < tiles <= 1280
    return tiles >= (115 if K <= 1024 else 256) and N > 128 and (N > 1024 or N % 256 > 0)


def _plain_operands(x: torch.Tensor, w: torch.Tensor) -> bool:
    return (here(x) and x.dim() == w.dim() == 2 and plain_call(x, w)
            and x.dtype == w.dtype == torch.bfloat16 and x.shape[1] % 64 == 0
            and x.shape[1] == w.shape[1] and x.shape[1] < DEPTH
            and x.is_contiguous() and w.is_contiguous()
            and w.device == x.device and x.data_ptr() % 16 == 0 and w.data_ptr() % 16 == 0)


def few_rows(x: torch.Tensor, w: torch.Tensor) -> bool:
    """Whether the kernels for few rows can take x [M, K] and w [N, K]."""
    return x.dim() == 2 and x.shape[0] <= FEW_ROWS and _plain_operands(x, w)


def _plain_bias(x: torch.Tensor, w: torch.Tensor, bias: torch.Tensor | None) -> bool:
    return (bias is None or plain_call(bias) and bias.dtype == x.dtype
            and bias.device == x.device and bias.shape == w.shape[:1] and bias.is_contiguous())


def linear_route(M: int, N: int, K: int) -> str | None:
    """Which of the extension's products is the faster way for x [M, K] and w [N, K]; None where
    the library is."""
    if M <= FEW_ROWS and rows_pay(M, N, K):
        return "linear_rows"
    if M > FEW_ROWS and blocks_pay(M, N, K):
        return "linear_blocks"
    if mid_pays(M, N, K):
        return "linear_mid"
    return "linear_big" if N % 4 == 0 and K < 1 << 22 and big_pays(M, N, K) else None


def linear_kernel(x: torch.Tensor, w: torch.Tensor, bias: torch.Tensor | None) -> str | None:
    """Which of the extension's products takes these, None where it is the library."""
    if x.dim() != 2 or w.dim() != 2:
        return None
    name = linear_route(x.shape[0], *w.shape)
    if name is None or not _plain_operands(x, w) or not _plain_bias(x, w, bias):
        return None
    if name in ("linear_mid", "linear_big") and x.shape[1] == 0:
        return None
    if name == "linear_big" and bias is not None and bias.data_ptr() % 4:
        return None
    return name


def linear_by(name: str | None, x: torch.Tensor, w: torch.Tensor,
              bias: torch.Tensor | None) -> torch.Tensor:
    """x w^T + bias by what linear_kernel said of them."""
    if name is None:
        return F.linear(x, w, bias)
    if name == "linear_mid":
        return linear_ext().linear_mid(x, w, None, None, bias)
    return getattr(linear_ext(), name)(x, w, bias)


def linear_takes_big(x: torch.Tensor, w: torch.Tensor, bias: torch.Tensor | None) -> bool:
    """Whether linear takes these to linear_big."""
    return linear_kernel(x, w, bias) == "linear_big"


def linear(x: torch.Tensor, w: torch.Tensor, bias: torch.Tensor | None = None,
           routed: bool = False) -> torch.Tensor:
    """x w^T + bias.  `routed`: a router reads what becomes of it.  A token's experts hang on
    near ties of the router's logits, and other last bits turn one of them in a token of some
    thousand (a prompt's logits 0.046 off in place of 0.015), so more rows than few are left to
    the library, with whose bits such models were checked.  It is no nearer to 64 bits than the
    kernels, and other numbers of rows, as of a prompt in portions, have other bits by it too."""
    if routed and (x.dim() != 2 or x.shape[0] > FEW_ROWS):
        return F.linear(x, w, bias)
    name = linear_kernel(x, w, bias)
    return linear_by(None if routed and name != "linear_rows" else name, x, w, bias)


def linear_parts(x: torch.Tensor, w: torch.Tensor, bias: torch.Tensor | None = None):
    """x w^T + bias for a kernel that can add up parts as it reads them: [M, N], or, where
    the depth is divided among workgroups, float32 parts [parts, M, N] of x w^T without the
    bias.  See sum_parts for what they stand for."""
    name = linear_kernel(x, w, bias)
    if name == "linear_rows":
        return linear_ext().linear_rows_parts(x, w, bias)
    return linear_by(name, x, w, bias)


def sum_parts(y: torch.Tensor, dtype: torch.dtype,
              bias: torch.Tensor | None = None) -> torch.Tensor:
    """What linear_parts' result stands for."""
    if y.dim() == 2:
        return y
    s = y[0]
    for p in y[1:]:
        s = s + p
    return (s if bias is None else s + bias.float()).to(dtype)
