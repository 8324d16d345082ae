"""Mixture of experts, and the grouped products it is made of.

A token's experts are chosen by a 32-bit router; each expert runs over the list
of its tokens (gathered on the way in, scattered to [token, choice] rows on the
way out), so no step's launch depends on how many tokens an expert got and the
whole can be captured in a graph.  The choices' rows are added by the next norm
in their order.

GPU: csrc/moe.hip."""
from __future__ import annotations

import torch
import torch.nn.functional as F

from . import serve_ext
from .linear import here, plain_call

# Rows up to which separate GEMMs cost more than one launch, whatever the sizes.  With more
# one launch of whole steps of the depth, if there are a few products of them, and either not
# too deep, for without enough tiles for the CUs the library divides the depth, or filling
# csrc/gemm_big.h's tiles.  us, one launch / library calls (and 20 us each on the host):
#   4 of 1536 x 1536   300 rows 23 / 33   700 28 / 48   1200 30 / 54   4000 67 / 83   12000 182 / 221
#   4 of 512 x 512     300 rows 6 / 20    4 of 320 x 2048   700 rows 27 / 34, 12000 88 / 92
#   4 of 4096 x 4096   300 rows 60 / 84 (not filled)   700 78 / 112   4000 373 / 350   12000 1158 / 1772
#   4 of 256 x 4096    700 rows 48 / 41   8 of 320 x 4096   300 rows 48 / 72, 12000 375 / 421
#   4 of 1536 x 6144   260 rows 73 / 72   2 of 512 x 2048   700 rows 27 / 19
#   2 of 1536 x 1536   260 rows 21 / 15   2 of 256 x 4096   700 rows 48 / 21
#   1 of 4096 x 4096   260 rows 48 / 21, 4000 94 / 89
STACKED_ROWS = 256
STACKED_PRODUCTS = 4
STACKED_DEPTH = 512         # for each product


def group_linear(x: torch.Tensor, w: torch.Tensor,
                 out: torch.Tensor | None = None) -> torch.Tensor:
    """x [T, G, K], w [G, N, K] -> [T, G, N]: a linear of its own for every
    group (head).  x and out may be strided in T and G, w in G."""
    if out is None:
        out = torch.empty(x.shape[0], w.shape[0], w.shape[1], dtype=x.dtype, device=x.device)
    if x.is_cuda:
        serve_ext().group_linear(x, w, out)
        return out
    return out.copy_(torch.einsum("tgk,gnk->tgn", x.float(), w.float()))


def _stacks(x: torch.Tensor, w: torch.Tensor) -> bool:
    return (here(x) and plain_call(x, w) and x.dim() == w.dim() == 3 and x.dtype == w.dtype
            and w.device == x.device and STACKED_PRODUCTS <= x.shape[0] == w.shape[0] <= 64
            and x.shape[2] == w.shape[2] and x.shape[2] % 64 == 0 and w.shape[1] % 4 == 0
            and w.shape[1] >= 256 and x.is_contiguous() and w.is_contiguous()
            and x.data_ptr() % 16 == 0 and w.data_ptr() % 16 == 0
            and x.shape[1] * x.shape[2] < 1 << 30
            and (x.shape[2] <= STACKED_DEPTH * x.shape[0] or serve_ext().group_linear_fills(
                x.shape[1], x.shape[0], w.shape[1], x.shape[2])))


def stacked_linear(x: torch.Tensor, w: torch.Tensor):
    """x [G, T, K], w [G, N, K] -> G results [T, N]: one launch while the rows
    are few, or the kernel for many takes them."""
    if x.is_cuda and x.dtype == torch.bfloat16 and (
            x.shape[1] <= STACKED_ROWS or _stacks(x, w)):
        out = torch.empty(x.shape[0], x.shape[1], w.shape[1], dtype=x.dtype, device=x.device)
        group_linear(x.transpose(0, 1), w, out.transpose(0, 1))
        return out
    return [F.linear(a, b) for a, b in zip(x, w)]


def moe_route(h: torch.Tensor, router: torch.Tensor, bias: torch.Tensor, top: int):
    """z = router h + bias in 32-bit; the `top` largest (the lower index wins a
    tie) and the softmax over them.

    Returns chosen [T, top] int32, weights [T, top] float32, lists [E, T] int32
    and counts [E] int32: lists[e, :counts[e]] are the rows t * top + choice
    that use expert e, in order."""
    if h.is_cuda:
        return serve_ext().moe_route(h, router, bias, top)
    T, E = h.shape[0], router.shape[0]
    z = h.float() @ router.float().T + bias.float()
    v, chosen = torch.sort(z, dim=-1, descending=True, stable=True)
    chosen = chosen[:, :top].int()
    weights = torch.softmax(v[:, :top], dim=-1)
    lists = torch.zeros(E, T, dtype=torch.int32)
    counts = torch.zeros(E, dtype=torch.int32)
    for e in range(E):
        rows = (chosen.flatten() == e).nonzero(as_tuple=True)[0]
        lists[e, :len(rows)] = rows.int()
        counts[e] = len(rows)
    return chosen, weights, lists, counts


def moe_experts(h: torch.Tensor, gate_up: torch.Tensor, down: torch.Tensor, routing):
    """h [T, W]; gate_up [E, 2, ff, W], down [E, W, ff].  Returns [T, top, W]:
    each choice's down(silu(gate h) * (up h)) times its weight."""
    chosen, weights, lists, counts = routing
    T, top = chosen.shape
    if h.is_cuda:
        ext = serve_ext()
        act = ext.moe_gate_up(h, gate_up, lists, counts, top)
        return ext.moe_down(act, down, lists, counts, weights)
    y = torch.zeros(T * top, h.shape[1])
    for e in range(counts.shape[0]):
        rows = lists[e, :int(counts[e])].long()
        g, u = (h[rows // top].float() @ gate_up[e, i].float().T for i in (0, 1))
        a = (torch.nn.functional.silu(g) * u).to(h.dtype).float()
        y[rows] = (a @ down[e].float().T) * weights.flatten()[rows, None]
    return y.view(T, top, -1).to(h.dtype)
