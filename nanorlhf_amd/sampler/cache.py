"""What the engine keeps of live sequences: KV pages and state slots.

Attention layers keep keys and values of every token (or the latent vector
both are made from) in pages, sized against 288 GB HBM3E; a sequence owns a
list of pages.  Recurrent layers keep one 32-bit matrix per head, and where
they need it their last input, in a slot; a sequence owns one slot number,
valid in every such layer.  A layer that runs several times in one forward has
an entry, with memory of its own, for every time.  Pages and slot are recycled
when a sequence finishes (continuous batching admits queued sequences into the
freed space).  Neither is cleared: keys beyond a sequence's length are never
visible, and a sequence's first token starts from a zero state."""
from __future__ import annotations

import numpy as np
import torch

from ..ops import serve_ext
from ..models.config import KVSpec, LatentSpec, StateSpec


class PagedKVCache:
    """layers[i] is (K, V) of an attention layer, [num_pages, page_size, heads,
    k_dim] and d-major per page [num_pages, heads, v_dim, page_size] (so the
    decode kernel's PV MFMA B-fragment is a contiguous 16-B load); the latents
    of a latent-attention layer, [num_pages, page_size, width]; or the state of
    a recurrent layer, [num_slots, heads, dim, vdim] float32, with its last
    input [num_slots, shift] beside it if it keeps one."""

    def __init__(self, cfg, num_pages: int, page_size: int = 16, device="cpu",
                 dtype=torch.bfloat16, num_slots: int = 0):
        self.page_size = page_size
        self.num_pages = num_pages
        self.device = device
        specs = cfg.cache_layers()
        self.stateful = any(isinstance(s, StateSpec) for s in specs)
        self.num_slots = num_slots if self.stateful else 0
        if self.stateful and num_slots < 1:
            raise ValueError("a model with recurrent layers needs state slots")
        self.layers = [self._make(s, dtype) for s in specs]
        self._free = list(range(num_pages - 1, -1, -1))
        self._free_slots = list(range(self.num_slots - 1, -1, -1))

    def _make(self, s, dtype):
        def zeros(*shape, dt=dtype):
            return torch.zeros(shape, dtype=dt, device=self.device)

        if isinstance(s, KVSpec):
            return (zeros(self.num_pages, self.page_size, s.heads, s.k_dim),
                    zeros(self.num_pages, s.heads, s.v_dim, self.page_size))
        if isinstance(s, LatentSpec):
            return zeros(self.num_pages, self.page_size, s.width)
        state = zeros(self.num_slots, s.heads, s.dim, s.vdim, dt=torch.float32)
        return (state, zeros(self.num_slots, s.shift)) if s.shift else state

    @property
    def free_pages(self) -> int:
        return len(self._free)

    @property
    def free_slots(self) -> int:
        return len(self._free_slots)

    def alloc(self, n: int) -> list[int]:
        if n > len(self._free):
            raise RuntimeError(f"KV pool exhausted: want {n}, have {len(self._free)} pages")
        return [self._free.pop() for _ in range(n)]

    def free(self, pages: list[int]):
        self._free.extend(pages)

    def copy_prompts(self, pairs: list[tuple["SeqState", "SeqState"]]):
        """For each (have, want) the pages of have's tokens, copied to want's."""
        n = [-(-len(a) // self.page_size) for a, _ in pairs]
        src, dst = (torch.tensor([p for pair, k in zip(pairs, n) for p in pair[i].pages[:k]],
                                 dtype=torch.int32, device=self.device) for i in (0, 1))
        pools = [t for layer in self.layers for t in layer]
        if src.is_cuda:
            serve_ext().copy_pages(pools, src, dst)
        else:
            for t in pools:
                t[dst.long()] = t[src.long()]

    def release(self, seq: "SeqState"):
        """Give back everything a sequence holds."""
        self.free(seq.pages)
        seq.pages = []
        if seq.state_slot >= 0:
            self._free_slots.append(seq.state_slot)
            seq.state_slot = -1

    @staticmethod
    def bytes_per_token(cfg, dtype=torch.bfloat16) -> int:
        width = {KVSpec: lambda s: s.heads * (s.k_dim + s.v_dim),
                 LatentSpec: lambda s: s.width, StateSpec: lambda s: 0}
        return sum(width[type(s)](s) for s in cfg.cache_layers()) * dtype.itemsize

    @staticmethod
    def bytes_per_slot(cfg, dtype=torch.bfloat16) -> int:
        return sum(4 * s.heads * s.dim * s.vdim + dtype.itemsize * s.shift
                   for s in cfg.cache_layers() if isinstance(s, StateSpec))

    @classmethod
    def for_budget(cls, cfg, max_tokens_total: int, page_size: int = 16, device="cpu",
                   dtype=torch.bfloat16, num_slots: int = 0) -> "PagedKVCache":
        pages = (max_tokens_total + page_size - 1) // page_size
        return cls(cfg, pages, page_size, device, dtype, num_slots)


class SeqState:
    """Book-keeping for one in-flight sequence."""

    __slots__ = ("uid", "tokens", "prompt_len", "pages", "finished", "out_index",
                 "logprobs", "computed", "state_slot")

    def __init__(self, uid: int, prompt: list[int], out_index: int):
        self.uid = uid
        self.tokens = list(prompt)
        self.prompt_len = len(prompt)
        self.pages: list[int] = []
        self.finished = False
        self.out_index = out_index
        self.logprobs: list[float] = []  # per generated (response) token
        self.computed = 0        # tokens whose KV and state the cache holds
        self.state_slot = -1

    def __len__(self):
        return len(self.tokens)

    @property
    def response(self) -> list[int]:
        return self.tokens[self.prompt_len:]

    def slot_of(self, pos: int, page_size: int) -> int:
        return self.pages[pos // page_size] * page_size + pos % page_size

    def slots_for(self, start: int, end: int, page_size: int) -> np.ndarray:
        pos = np.arange(start, end)
        pages = np.asarray(self.pages, dtype=np.int64)
        return pages[pos // page_size] * page_size + pos % page_size

    def ensure_capacity(self, pool: PagedKVCache, upto: int):
        """Pages for `upto` tokens, and a state slot if the model keeps states."""
        if pool.stateful and self.state_slot < 0:
            if not pool._free_slots:
                raise RuntimeError("no free state slot")
            self.state_slot = pool._free_slots.pop()
        need = (upto + pool.page_size - 1) // pool.page_size
        if need > len(self.pages):
            self.pages.extend(pool.alloc(need - len(self.pages)))
