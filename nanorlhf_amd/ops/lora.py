"""Fused LoRA linear: y = x·Wᵀ + (α/r)·(x·Aᵀ)·Bᵀ + bias in ONE MFMA GEMM.

Replaces the 3-launch F.linear chain (reference peft call site
GRPO/grpo.py:226-243).  The adapter contribution rides as one extra K-tile of the
base GEMM (csrc/lora.hip), so the fused kernel does ≈(H+64)/H of the base GEMM's work
in a single launch.

Backward (W frozen under LoRA — no dW GEMM at all):
    du = s·(dy·B)            [M,r]   (_down)
    dx = dy·W + du·A         = the SAME kernel on (dy, Wᵀ) + (du, Aᵀ)
    dA = duᵀ·x               [r,H]   } one launch of csrc/lora_grad.hip
    dB = dyᵀ·u               [N,r]   }
Wᵀ is cached once per linear (W never changes while LoRA trains).

Constraints for the fused path: K % 64 == 0, rank == 64 (the reference
default, grpo.py:92); anything else falls back to the chained form.
"""
from __future__ import annotations

from typing import Optional

import torch

from . import ext
from .linear import DEPTH, mid_fills, one_round_of_blocks


def lora_gemm_ref(x, w, u=None, b=None, bias=None):
    """CPU/fp32 oracle of csrc/lora.hip::lora_gemm."""
    y = x.float() @ w.float().t()
    if u is not None:
        y = y + u.float() @ b.float().t()
    if bias is not None:
        y = y + bias.float()
    return y.to(x.dtype)


# Strategy cache: weight shape (N, K) -> {(edge of lora_gemm's tiles, whether they are many,
# whether there is a bias, device): "fused" | "epilogue"}.
# "fused"    = the single wide-K MFMA kernel (wins when our GEMM rate is
#              within the fusion savings of hipBLASLt — e.g. N-heavy shapes);
# "epilogue" = hipBLASLt base GEMM + the custom rank-64 lora_add_ MFMA pass
#              (wins on deep K: few rows, which the library divides, by far).
# They round y differently (the fused kernel once, the epilogue twice), so a choice that
# the timer's noise could turn would give a step other bits in another process.  One of them
# is the rule and the other has to be clearly faster: the fused kernel up to DEEP, where
# the epilogue's pass over y costs more than a tenth of the product (448 / K of it: y twice
# at 5.8 TB/s, the product at 1.3 PFLOP/s), the epilogue beyond, where they come close.
# 46673 rows, fused / epilogue in us: 1536 x 1536 241 / 296, 2048 x 1536 250 / 330, 17920 x
# 1536 2205 / 2610; 1536 x 8960 1020 / 1069, 1536 x 17920 1990 / 2015.
# Measured once per key on first touch (events, ~1 ms): up to 128 rows, which run in
# another kernel, say nothing about more, nor do a few tiles about many that fill the CUs, nor
# a square weight's dx, which has no bias, about its y.
_TUNE: dict[tuple, dict] = {}
DEEP = 4096


def _time_cuda(fn, reps: int = 3) -> float:
    fn()  # warm
    s, e = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    s.record()
    for _ in range(reps):
        fn()
    e.record()
    e.synchronize()
    return s.elapsed_time(e) / reps


def _capturing(x) -> bool:
    return x.is_cuda and torch.cuda.is_current_stream_capturing()


def _strategy_key(M, N, K, bias, device):
    return (ext().lora_gemm_tiles(M, K), ext().lora_gemm_big(M, N, K), bias is not None, device)


def _choose_strategy(x, w, u, b, bias) -> str:
    N, K = int(w.size(0)), int(w.size(1))
    M = x.shape[0]
    known = _TUNE.setdefault((N, K), {})
    key = _strategy_key(M, N, K, bias, x.device)
    st = known.get(key)
    if st is None and _capturing(x):            # nothing can be timed now
        return next(iter(known.values()), "fused" if K <= DEEP else "epilogue")
    if st is None:
        t_fused = _time_cuda(lambda: ext().lora_gemm(x, w, u, b, bias))

        def ep():
            y = torch.nn.functional.linear(x, w, bias)
            ext().lora_add_(y, u, b)
        t_ep = _time_cuda(ep)
        st = "fused" if t_fused <= (1.1 if K <= DEEP else 0.9) * t_ep else "epilogue"
        known[key] = st
    return st


def _mid(M: int, N: int, K: int) -> bool:
    """Whether lora_gemm takes csrc/linear_mid.hip's tiles of 128.  Library and lora_add_ / these in
    us, over operands that no cache holds: 1000 rows of 896 x 896 13.3 / 11.4, 2667 17.5 / 11.7,
    1800 of 2048 x 1536 25.5 / 19.4, 2667 of 1536 x 2048 31 / 24 (tiles of 256 27 to 33), 100 of
    17920 x 1536 30 / 22; the slowest 2667 of 512 x 2048 20.9 / 22.7.  Deeper the library divides
    what is no round, 1300 of 896 x 4864 34 / 47, 1800 of 1536 x 8960 73 / 81, 1000 and 2667 of
    1536 x 12288 74 / 113 and 121 / 119, of 1536 x 16384 91 / 138 and 152 / 149, up to a depth from
    which it takes kernels of half the rate: of 1536 x 17920 200 / 160 and 214 / 161, of 2048 x
    18944 199 / 165 (1800 rows 219 / 169), 1300 of 1536 x 37888 312 / 323, 1152 of 3584 x
    18944 225 / 174; but 800 of 2048 x 17920 133 / 157 and 1800 of 896 x 17920 130 / 158.  What is
    left between is timed."""
    if K <= 2048:
        return mid_fills(M, N, 0.0)
    return 16384 < K < 1 << 22 and M >= 1000 and N >= 1024 and mid_fills(M, N, 0.375)


def one_round(M: int, N: int, K: int) -> int:
    """The edge of the tiles, 64 or 128, in which lora_gemm takes the product in one round of the
    CUs; 0 where it does not.  csrc/lora.hip lora_gemm_round is the same rule.  Blocks of 64 also
    of many rows of a few columns, for which the library needs a pass more: library and
    lora_add_ / tiles of 128 / blocks in us, of a depth of 896: 1200 x 64 11.8 / 10.5 / 5.0, 16384 x
    64 18.4 / 12.6 / 11.6, 2048 x 512 13.6 / 11.2 / 9.7; of 2048 4000 x 128 20 / 23 / 13."""
    return 64 if one_round_of_blocks(M, N) and K < DEPTH else 128 if _mid(M, N, K) else 0


def _dispatch_gemm(x, w, u, b, bias):
    """y = x·wᵀ + u·bᵀ (+bias) via the per-shape-tuned strategy, or in blocks of 64 rows
    (csrc/linear_rows.hip) while they are one round of the CUs.  212 rows, library and
    lora_add_ / blocks in us: 1152 x 896 9.5 / 5.5, 1536 x 8960 30 / 23, 1536 x 17920 81 / 43
    (tiles of 256 13 to 20 at a depth of 896 and 1536, 55 at 4864); 66 of 896 x 9728 16 / 19,
    with the host's share 22 / 20.  More rows take tiles of 128 (_mid)."""
    st = _known_strategy(x, w, bias) or _choose_strategy(x, w, u, b, bias)
    if st == "fused":
        return ext().lora_gemm(x, w, u, b, bias)
    y = torch.nn.functional.linear(x, w, bias)
    if not y.is_contiguous():
        y = y.contiguous()
    ext().lora_add_(y, u, b)
    return y


def _known_strategy(x, w, bias) -> str | None:
    """The strategy that a rule says or an earlier call measured, None if neither does.  A
    rule's answer is not put among the measured ones: its sizes have no key of their own."""
    M, (N, K) = x.shape[0], w.shape
    known = _TUNE.setdefault((N, K), {})
    if one_round(M, N, K):
        return "fused"
    return known.get(_strategy_key(M, N, K, bias, x.device)) if known else None


# Products down to the rank are csrc/lora_grad.hip's lora_down, unless both many rows
# and many columns, where the library streams them 5 to 20% faster.  Library against
# kernel, in us: 240 x 896 14 / 7, 4096 x 8960 43 / 25, 8000 x 3584 22 / 21, 48720 x 1536
# 38 / 37; 16000 x 3584 28 / 32, 24000 x 8960 93 / 112, 64000 x 2048 58 / 65.
DOWN_ROWS, DOWN_COLS, DOWN_SIZE = 8192, 2048, 100_000_000
# Gradients of more columns than these leave no room to divide the tokens evenly: 16000
# tokens of 37888 columns 247 / 284 us, 240 tokens 13.4 / 9.4.
GRAD_COLS, GRAD_ROWS = 20480, 512


def _fast_down(z: torch.Tensor, p: torch.Tensor, flat: bool) -> bool:
    """Whether csrc/lora_grad.hip's lora_down takes z and p, and not a backward that is itself
    recorded."""
    C = z.shape[1]
    return (z.shape[0] <= DOWN_ROWS or C <= DOWN_COLS and z.numel() <= DOWN_SIZE) \
        and C % (64 if flat else 8) == 0 and z.dtype == p.dtype == torch.bfloat16 \
        and p.shape[0 if flat else 1] == 64 and not torch.is_grad_enabled()


def _down(z: torch.Tensor, p: torch.Tensor, scale: float, flat: bool) -> torch.Tensor:
    """scale * z pᵀ with p [r, C] (flat), or scale * z p with p [C, r]; the scale rides
    on the product's sums."""
    if _fast_down(z, p, flat):
        return ext().lora_down(z.contiguous(), p.contiguous(), scale, flat)
    return torch.addmm(z.new_empty(1), z, p.t() if flat else p, beta=0, alpha=scale)


def _fast_grad(z: torch.Tensor) -> bool:
    """Whether csrc/lora_grad.hip's lora_grads takes the gradient with z [M, C] in it, and
    not a backward that is itself recorded."""
    return z.shape[1] % 8 == 0 and z.dtype == torch.bfloat16 and not torch.is_grad_enabled() \
        and (z.shape[1] <= GRAD_COLS or z.shape[0] <= GRAD_ROWS)


def _forward(x, w, bias, lora_A, lora_B, scaling):
    """(y, u): the product with its adapter and the adapter's x down to the rank."""
    st = _known_strategy(x, w, bias) if x.dim() == 2 and _fast_down(x, lora_A, True) else None
    if st is not None:
        return ext().lora_forward(x, w, bias, lora_A, lora_B, scaling, st == "fused")
    # u = s·x·Aᵀ (skinny GEMM, r=64)
    u = _down(x, lora_A, scaling, True)
    return _dispatch_gemm(x.contiguous(), w, u, lora_B.contiguous(), bias), u


def _backward(dy, x, u, lora_A, lora_B, w_t, scaling, want_x, want_A, want_B):
    """(dx, dA, dB), None for those that are not wanted."""
    if dy.dim() == 2 and _fast_down(dy, lora_B, False) and lora_A.shape[1] % 64 == 0 \
            and (not want_A or _fast_grad(x)) and (not want_B or _fast_grad(dy)):
        st = _known_strategy(dy, w_t, None) if want_x else "fused"
        if st is not None:
            return ext().lora_backward(dy, x, u, lora_A, lora_B, w_t, scaling,
                                       st == "fused", want_x, want_A, want_B)
    dy = dy.contiguous()
    # du = s·dy·B  [M, r]
    du = _down(dy, lora_B, scaling, False)
    dx = None
    if want_x:
        # dx = dy·W + du·A → same dispatch on (dy, Wᵀ) + (du, Aᵀ)
        a_t = lora_A.t().contiguous()
        dx = _dispatch_gemm(dy, w_t, du, a_t, None)
    if not (want_A or want_B):
        return dx, None, None
    fast_A, fast_B = want_A and _fast_grad(x), want_B and _fast_grad(dy)
    dA = dB = None
    if fast_A or fast_B:
        dA, dB = ext().lora_grads(
            *((x.contiguous(), du.contiguous()) if fast_A else (None, None)),
            *((dy, u.contiguous()) if fast_B else (None, None)))
    if want_A and not fast_A:
        dA = du.t() @ x
    if want_B and not fast_B:
        dB = dy.t() @ u
    return dx, dA if want_A else None, dB if want_B else None


class _FusedLoRAFn(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, w, bias, lora_A, lora_B, scaling, w_t_cache):
        y, u = _forward(x, w, bias, lora_A, lora_B, scaling)
        ctx.save_for_backward(x, u, lora_A, lora_B, w_t_cache)
        ctx.scaling = scaling
        return y

    @staticmethod
    def backward(ctx, dy):
        want_x, (want_A, want_B) = ctx.needs_input_grad[0], ctx.needs_input_grad[3:5]
        dx, dA, dB = _backward(dy, *ctx.saved_tensors, ctx.scaling, want_x, want_A, want_B)
        return dx, None, None, dA, dB, None, None


def glu_keeps(M: int, N: int, K: int) -> bool:
    """Whether a gate/up product of these sizes writes its activation too (csrc/lora.hip
    lora_glu): where its kernel is the one of 256-tiles anyway, which is to say more than 128
    rows that one_round does not take, up to a depth of 2048.  Product and pass / lora_glu over
    700, 2667 and 13000 rows of 17920 to 37888: 1.02 (0.97, 1.07) at 2048, 1.00 (0.97, 1.07) at
    2560, 3072 and 3584."""
    return M > 128 and N % 8 == 0 and K <= 2048 and not one_round(M, N, K)


class _LoRAGluFn(torch.autograd.Function):
    """swiglu of _FusedLoRAFn's y [T, 2 I] without a bias."""

    @staticmethod
    def forward(ctx, x, w, lora_A, lora_B, scaling, w_t_cache):
        act = None
        if glu_keeps(x.shape[0], *w.shape):
            u, x2, b = _down(x, lora_A, scaling, True), x.contiguous(), lora_B.contiguous()
            st = _known_strategy(x2, w, None) or _choose_strategy(x2, w, u, b, None)
            if st == "fused":
                act, kept = ext().lora_glu(x2, w, u, b)
            else:
                kept = _dispatch_gemm(x2, w, u, b, None)
        else:
            kept, u = _forward(x, w, None, lora_A, lora_B, scaling)
        if act is None:
            act = ext().swiglu_fwd(kept)
        ctx.save_for_backward(x, u, lora_A, lora_B, w_t_cache, kept)
        ctx.scaling = scaling
        return act

    @staticmethod
    def backward(ctx, dact):
        *saved, kept = ctx.saved_tensors
        want_x, (want_A, want_B) = ctx.needs_input_grad[0], ctx.needs_input_grad[2:4]
        dx, dA, dB = _backward(ext().swiglu_bwd(dact.contiguous(), kept), *saved, ctx.scaling,
                               want_x, want_A, want_B)
        return dx, None, dA, dB, None, None


def fused_lora_linear(x: torch.Tensor, w: torch.Tensor,
                      bias: Optional[torch.Tensor],
                      lora_A: torch.Tensor, lora_B: torch.Tensor,
                      scaling: float, w_t_cache: torch.Tensor) -> torch.Tensor:
    """x: [T, K]; w: [N, K] frozen; lora_A: [r, K]; lora_B: [N, r]."""
    return _FusedLoRAFn.apply(x, w, bias, lora_A, lora_B, scaling, w_t_cache)


def fused_lora_glu(x: torch.Tensor, w: torch.Tensor, lora_A: torch.Tensor,
                   lora_B: torch.Tensor, scaling: float,
                   w_t_cache: torch.Tensor) -> torch.Tensor:
    """swiglu(fused_lora_linear(x, w, None, ...)) of w's gate rows, then up rows."""
    return _LoRAGluFn.apply(x, w, lora_A, lora_B, scaling, w_t_cache)


def fused_path_ok(w: torch.Tensor, r: int) -> bool:
    return (w.is_cuda and w.dtype == torch.bfloat16 and r == 64
            and w.size(1) % 64 == 0)
