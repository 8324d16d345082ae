"""Embedding lookup whose weight is trained."""
from __future__ import annotations

import torch
import torch.nn.functional as F

from . import ext
from .linear import here, plain_call, unwatched

# Tokens up to which the kernel compares all ids with each other, which grows with their square;
# torch sorts from 3072 on.  torch / kernel in us, over random ids and with a third of the tokens
# of one id: 4096 x 1536 of 152 thousand rows 168 / 98 and 172 / 166, 6000 200 / 117 and 203 / 214.
# What adds up one id's tokens is one workgroup: of 16384 rows 4096 x 1536 with a tenth of one id 97 /
# 43, with all of them 180 / 293, 4096 x 3584 148 / 44 with none, 144 / 207 with a third.
KERNEL_TOKENS = 4096


class _EmbeddingFn(torch.autograd.Function):
    @staticmethod
    def forward(ctx, ids, weight):
        ctx.save_for_backward(ids)
        ctx.rows = weight.shape[0]
        return F.embedding(ids, weight)

    @staticmethod
    def backward(ctx, dy):
        (ids,) = ctx.saved_tensors
        if torch.is_grad_enabled() or ids.shape[0] > KERNEL_TOKENS:     # a recorded backward
            return None, torch.ops.aten.embedding_dense_backward(dy, ids, ctx.rows, -1, False)
        dy = dy.contiguous()
        return None, ext().embedding_grad(ids, dy if dy.data_ptr() % 16 == 0 else dy.clone(),
                                          ctx.rows)


def embedding(ids: torch.Tensor, weight: torch.Tensor) -> torch.Tensor:
    """weight[ids]; the gradient of few tokens by the kernel, whose sums are 32-bit."""
    if torch.is_grad_enabled() and weight.requires_grad and here(weight) and ids.is_cuda \
            and ids.dim() == 1 and ids.dtype == torch.int64 and ids.is_contiguous() \
            and weight.dtype == torch.bfloat16 and weight.shape[1] % 8 == 0 \
            and not torch.is_autocast_enabled() and unwatched(ids, weight):
        return _EmbeddingFn.apply(ids, weight)
    return F.embedding(ids, weight)


def embed_rms_norm(ids: torch.Tensor, weight: torch.Tensor, norm: torch.Tensor, eps: float,
                   place: tuple | None = None):
    """[rms_norm(h, norm, eps), h = weight[ids]] in one launch, and with place (lengths, pages,
    page size) what decode_inputs says of it too; None where no kernel takes these."""
    if not (here(weight) and ids.is_cuda and ids.dim() == 1 and ids.dtype == torch.int64
            and ids.is_contiguous() and plain_call(ids, weight, norm)
            and weight.dtype == norm.dtype == torch.bfloat16 and weight.dim() == 2
            and weight.shape[1] % 8 == 0 and 0 < weight.shape[1] <= 8192
            and norm.numel() == weight.shape[1] and ids.device == norm.device == weight.device
            and all(t.is_contiguous() and t.data_ptr() % 16 == 0 for t in (weight, norm))):
        return None
    return ext().embed_rms_norm(ids, weight, norm, eps, *(place or ()))
