"""In-process generation engine — the vLLM replacement.

Deletes the reference's per-update disk round trip (save LoRA → reload base
→ merge_and_unload → save merged → boot LLM() → generate → del llm,
GRPO/grpo_trainer.py:122-166): here the sampler runs the live policy module
in-place (LoRA pre-merged into an HBM buffer, models/lora.py), with a paged
KV pool, continuous batching (finished sequences free pages, queued ones are
admitted), prefill via the varlen MFMA flash kernel and decode via the paged
LDS-staged attention kernel, temperature/top-p sampling in HIP.

API mirrors the reference's `vllm_generate(N, model, tokenizer, prompts,
temperature, max_tokens)` contract (grpo_trainer.py:122-166): `generate`
returns per-prompt responses padded to max_tokens with the pad token.
"""
from __future__ import annotations

from dataclasses import dataclass

import numpy as np
import torch

from .. import ops
from ..models.qwen2 import AttnContext, Portions
from ..models.lora import merge_for_rollout, unmerge
from .cache import PagedKVCache, SeqState
from .decode_batch import DecodeBatch


@dataclass
class SamplingParams:
    n: int = 1
    temperature: float = 1.0
    top_p: float = 0.95
    max_tokens: int = 128
    seed: int = 0
    stop_token_id: int | None = None  # EOS; None → run to max_tokens


class SamplerEngine:
    KV_DTYPES = {"bf16": torch.bfloat16, "fp8_e4m3": torch.float8_e4m3fn}

    # device memory that state slots may take unless state_slots says otherwise
    STATE_BYTES = 32 << 30

    def __init__(self, model, kv_pool_tokens: int, page_size: int = 16,
                 max_num_seqs: int = 4096, prefill_chunk_tokens: int = 131072,
                 compact_interval: int = 32, use_graphs: bool = True,
                 kv_cache_dtype: str = "bf16",
                 rollout_weight_dtype: str = "bf16",
                 state_slots: int | None = None):
        if kv_cache_dtype not in model.kv_cache_dtypes:
            raise ValueError(f"{type(model).__name__} caches {model.kv_cache_dtypes}, "
                             f"not {kv_cache_dtype!r}")
        self.model = model
        self.device = next(model.parameters()).device
        self.dtype = next(model.parameters()).dtype
        kv_dtype = (self.KV_DTYPES[kv_cache_dtype]
                    if self.device.type == "cuda" or kv_cache_dtype != "bf16"
                    else self.dtype)
        if kv_cache_dtype == "bf16":
            kv_dtype = self.dtype  # float32 models cache float32
        per_slot = PagedKVCache.bytes_per_slot(model.cfg, kv_dtype)
        if per_slot and state_slots is None:
            state_slots = max(1, min(max_num_seqs, self.STATE_BYTES // per_slot))
        self.pool = PagedKVCache.for_budget(model.cfg, kv_pool_tokens, page_size,
                                            device=self.device, dtype=kv_dtype,
                                            num_slots=state_slots or 0)
        self.max_num_seqs = max_num_seqs
        self.prefill_chunk_tokens = prefill_chunk_tokens
        self.compact_interval = compact_interval
        self.use_graphs = use_graphs and self.device.type == "cuda"
        self._graph = None
        self._graph_version = None
        self._step_dev = (torch.zeros(1, dtype=torch.long, device=self.device)
                          if self.device.type == "cuda" else None)
        # "fp8_e4m3": rollout-only e4m3 layer weights via torch._scaled_mm
        # (inference GEMMs at ~2x the bf16 rate; lm_head stays bf16 so the
        # sampled logits/logprobs come from the exact head).  Training
        # weights are never touched; validated like the fp8 KV mode.
        self.rollout_weight_dtype = (rollout_weight_dtype
                                     if self.device.type == "cuda" else "bf16")

    # ----------------------------------------------------------------- utils
    def _sample_from_hidden(self, hidden_last: torch.Tensor,
                            params: SamplingParams, counts: bool = True):
        """Returns (tokens [B], logprobs [B] fp32) — the chosen token's
        logprob under the temperature-scaled softmax (vLLM logprobs parity;
        matches the scoring pass's logits/temperature quirk)."""
        logits = self.model.logits(hidden_last)
        if self._step_dev is not None:
            # device-side step counter: correct under hipGraph replay; a decode step's
            # commit counts it
            if counts:
                self._step_dev.add_(1)
            tok, lp = ops.ext().sample_topp_dev(logits.contiguous(),
                                                float(params.temperature),
                                                float(params.top_p),
                                                int(params.seed), self._step_dev,
                                                0 if counts else 1)
            return tok, lp
        self._sample_step += 1
        tok = ops.sample_tokens(logits, params.temperature, params.top_p,
                                params.seed, self._sample_step)
        inv_t = 1.0 / params.temperature if params.temperature > 0 else 1.0
        logp = torch.log_softmax(logits.float() * inv_t, dim=-1)
        lp = logp.gather(1, tok.unsqueeze(1)).squeeze(1)
        return tok, lp

    # ----------------------------------------------------------------- step
    def _step_context(self, entries):
        """Batch description of one step: single tokens first, then portions.
        Returns (ids, ctx, first row of each entry)."""
        ps = self.pool.page_size
        order = sorted(range(len(entries)), key=lambda e: entries[e][1] != 1)
        nd = sum(n == 1 for _, n in entries)
        starts = [0] * len(entries)
        ids, pos, slots, row = [], [], [], 0
        for e in order:
            s, n = entries[e]
            a, b = s.computed, s.computed + n
            if n < 1 or b > len(s.tokens):
                raise ValueError(f"sequence {s.uid} has no tokens {a}..{b}")
            s.ensure_capacity(self.pool, b)
            starts[e] = row
            row += n
            ids.append(np.asarray(s.tokens[a:b], dtype=np.int64))
            pos.append(np.arange(a, b))
            slots.append(s.slots_for(a, b, ps))
        seqs = [entries[e][0] for e in order]
        lens = np.array([entries[e][1] for e in order])
        P = max(len(s.pages) for s in seqs)
        bt = np.zeros((len(seqs), P), dtype=np.int32)
        for r, s in enumerate(seqs):
            bt[r, :len(s.pages)] = s.pages
        ints = {"bt": bt, "slot": np.array([s.state_slot for s in seqs]),
                "len": np.array([s.computed for s in seqs]) + lens}
        if nd < len(seqs):
            plens = lens[nd:]
            cu = np.concatenate([[0], np.cumsum(plens)])
            per = -(-plens // ops.linear_attn.CHUNK)
            owner = np.repeat(np.arange(len(plens)), per)
            first = np.concatenate([[0], np.cumsum(per)])
            off = (np.arange(len(owner)) - first[owner]) * ops.linear_attn.CHUNK
            held = -(-ints["len"][nd:] // ops.linear_attn.CHUNK) * ops.linear_attn.CHUNK
            ctx_first = np.concatenate([[0], np.cumsum(held)])
            ints.update(ctx_first=ctx_first, cu=cu, row_seq=np.repeat(np.arange(len(plens)), plens),
                        fresh=np.array([s.computed == 0 for s in seqs[nd:]]),
                        chunks=np.stack([owner, cu[owner] + off,
                                         np.minimum(plens[owner] - off,
                                                    ops.linear_attn.CHUNK)]),
                        first=first)
        # one transfer for all int32 and one for all int64 arrays
        dev32 = torch.from_numpy(np.concatenate(
            [v.ravel() for v in ints.values()]).astype(np.int32)).to(self.device)
        t, at = {}, 0
        for k, v in ints.items():
            t[k] = dev32[at:at + v.size].view(v.shape)
            at += v.size
        ids, pos, slots = torch.from_numpy(np.stack(
            [np.concatenate(x) for x in (ids, pos, slots)])).to(self.device)
        ctx = AttnContext(mode="step", positions=pos, slots=slots, kv_caches=self.pool.layers)
        if nd:
            ctx.block_tables, ctx.seq_lens = t["bt"][:nd], t["len"][:nd]
            ctx.state_slots = t["slot"][:nd]
        if nd < len(seqs):
            ctx.portions = Portions(
                cu=t["cu"], seq_lens=t["len"][nd:], block_tables=t["bt"][nd:],
                row_seq=t["row_seq"], state_slots=t["slot"][nd:], fresh=t["fresh"],
                chunks=t["chunks"], chunk_first=t["first"], max_q=int(lens[nd:].max()),
                ctx_first=t["ctx_first"], keys=int(ctx_first[-1]),
                pairs=int((plens * ints["len"][nd:]).sum()))
        return ids, ctx, starts

    @torch.no_grad()
    def step(self, entries, on_layer=None):
        """Run the next n tokens of each (sequence, n), all as one batch, from
        what the cache holds of them; n == 1 is a decode step.

        Returns (hidden [tokens, width], starts): entry e's rows are
        starts[e] .. starts[e] + n - 1."""
        ids, ctx, starts = self._step_context(entries)
        ctx.on_layer = on_layer
        hidden = self.model(ids, ctx)
        for s, n in entries:
            s.computed += n
        return hidden, starts

    # -------------------------------------------------------------- prefill
    @torch.no_grad()
    def _prefill(self, seqs: list[SeqState], params: SamplingParams):
        """Run the prompts of `seqs` within the token budget of a batch and
        sample each one's first token.  Models with packed prefill run whole
        prompts; the others are cut wherever the budget ends."""
        if self.model.packed_prefill:
            return self._prefill_packed(seqs, params)
        todo = list(seqs)
        while todo:
            batch, room = [], self.prefill_chunk_tokens
            for s in todo:
                n = min(len(s) - s.computed, room)
                if n:
                    batch.append((s, n))
                    room -= n
            hidden, starts = self.step(batch)
            done = [(s, r + n - 1) for (s, n), r in zip(batch, starts) if s.computed == len(s)]
            if done:
                rows = torch.tensor([r for _, r in done], device=self.device)
                self._record_first([s for s, _ in done], hidden[rows], params)
            todo = [s for s in todo if s.computed < s.prompt_len]

    def _record_first(self, seqs, hidden, params):
        tokens, lps = self._sample_from_hidden(hidden, params)
        for s, t, l in zip(seqs, tokens.tolist(), lps.tolist()):
            s.tokens.append(int(t))
            s.logprobs.append(float(l))
            if params.stop_token_id is not None and int(t) == params.stop_token_id:
                s.finished = True

    def _prefill_packed(self, seqs: list[SeqState], params: SamplingParams):
        """Whole prompts as one packed varlen batch per token budget."""
        i = 0
        while i < len(seqs):
            chunk: list[SeqState] = []
            total = 0
            while i < len(seqs) and (not chunk or total + len(seqs[i]) <= self.prefill_chunk_tokens):
                total += len(seqs[i])
                chunk.append(seqs[i])
                i += 1
            # samples of one prompt run it once
            row, once, twins = {}, [], []
            for s in chunk:
                key = tuple(s.tokens)
                if key in row:
                    twins.append((once[row[key]], s))
                else:
                    row[key] = len(once)
                    once.append(s)
            lens = [len(s) for s in once]
            ids = torch.tensor([t for s in once for t in s.tokens], dtype=torch.long,
                               device=self.device)
            cu = torch.zeros(len(once) + 1, dtype=torch.int32, device=self.device)
            cu[1:] = torch.cumsum(torch.tensor(lens, dtype=torch.int32, device=self.device), 0)
            pos = torch.cat([torch.arange(n, device=self.device) for n in lens])
            slots = torch.from_numpy(np.concatenate(
                [s.slots_for(0, len(s), self.pool.page_size) for s in once])).to(self.device)
            ctx = AttnContext(mode="prefill", positions=pos, cu_seqlens=cu,
                              max_seqlen=max(lens), kv_caches=self.pool.layers, slots=slots)
            hidden = self.model(ids, ctx)[cu[1:].long() - 1]
            if twins:
                self.pool.copy_prompts(twins)
                hidden = hidden[torch.tensor([row[tuple(s.tokens)] for s in chunk],
                                             device=self.device)]
            for s in chunk:
                s.computed = len(s)
            self._record_first(chunk, hidden, params)

    # --------------------------------------------------------------- decode
    def _decode_step_eager(self, db: DecodeBatch, params: SamplingParams):
        hidden = self.model(db.last_tok, db.context(self.pool.layers))
        tokens, lps = self._sample_from_hidden(hidden, params, counts=False)
        db.commit(tokens, lps, self._step_dev)

    def _count_steps(self, n: int):
        """Sampling goes on as after n steps more."""
        if self._step_dev is not None:
            self._step_dev.add_(n)
        self._sample_step += n

    def _run_decode_step(self, db: DecodeBatch, params: SamplingParams,
                         left: int = 1 << 30) -> int:
        """One decode step; hipGraph-captured and replayed when the batch
        state is stable.  Returns the number of steps actually taken (capture
        does 2 warmup steps, so that with no more than those `left` there is none)."""
        stale = self._graph is None or self._graph_version != db.version
        if not self.use_graphs or stale and left <= 2:
            self._decode_step_eager(db, params)
            return 1
        if stale:
            torch.cuda.synchronize()
            side = torch.cuda.Stream()
            side.wait_stream(torch.cuda.current_stream())
            with torch.cuda.stream(side):
                for _ in range(2):
                    self._decode_step_eager(db, params)
            torch.cuda.current_stream().wait_stream(side)
            torch.cuda.synchronize()
            g = torch.cuda.CUDAGraph()
            with torch.cuda.graph(g):
                self._decode_step_eager(db, params)
            self._graph = g
            self._graph_version = db.version
            return 2  # the warmup steps ran; captured step executes on replay
        self._graph.replay()
        return 1

    # -------------------------------------------------------------- generate
    @torch.no_grad()
    def generate(self, prompts: list[list[int]], params: SamplingParams,
                 pad_token_id: int = 0, merge_lora: bool = True,
                 return_logprobs: bool = False):
        """Sample params.n continuations per prompt.

        Returns LongTensor [len(prompts)*n, max_tokens]: responses
        right-padded with pad_token_id, matching the reference's
        vllm_generate output contract (grpo_trainer.py:152-164).
        Row order: prompt-major (prompt0 sample0..n-1, prompt1 ...).
        """
        was_training = self.model.training
        self.model.eval()
        if merge_lora:
            merge_for_rollout(self.model,
                              quant=(self.rollout_weight_dtype
                                     if self.rollout_weight_dtype != "bf16" else None))
        try:
            waiting: list[SeqState] = []
            uid = 0
            for pi, p in enumerate(prompts):
                for j in range(params.n):
                    waiting.append(SeqState(uid, p, out_index=pi * params.n + j))
                    uid += 1
            done: list[SeqState] = []
            self._sample_step = 0
            if self._step_dev is not None:
                self._step_dev.zero_()
            self._graph = None  # new rollout -> new capture
            db = DecodeBatch(self.pool, [], params.max_tokens,
                             params.stop_token_id, self.device)
            outer_guard = 0

            def admit():
                """Move waiting → active, allocating each sequence's full page
                budget (prompt + max_tokens) up front: no oversubscription, so
                decode can never dead-lock on pages mid-flight."""
                admitted = []
                while waiting and len(db) + len(admitted) < self.max_num_seqs:
                    s = waiting[-1]
                    ps = self.pool.page_size
                    need = (len(s) + params.max_tokens + ps - 1) // ps
                    if need > self.pool.num_pages:
                        raise RuntimeError(
                            f"sequence needs {need} pages (prompt {len(s)} + "
                            f"max_tokens {params.max_tokens}) but the KV pool "
                            f"has only {self.pool.num_pages}; raise "
                            "kv_pool_tokens or lower response_length")
                    if need > self.pool.free_pages or (
                            self.pool.stateful and not self.pool.free_slots):
                        break
                    waiting.pop()
                    s.ensure_capacity(self.pool, len(s) + params.max_tokens)
                    admitted.append(s)
                return admitted

            while waiting or len(db):
                fresh = admit()
                if fresh:
                    self._prefill(fresh, params)
                    db.extend(fresh)
                # device-resident decode: no host sync inside the chunk, which ends where
                # every row has its tokens.  What is sampled after it is sampled as after a
                # whole chunk.
                inner, left = 0, min(self.compact_interval, db.steps_left())
                while len(db) and inner < left:
                    n = self._run_decode_step(db, params, db.steps_left())
                    inner, db.clock = inner + n, db.clock + n
                if waiting and len(db) and inner < self.compact_interval:
                    self._count_steps(self.compact_interval - inner)
                done.extend(db.compact())
                outer_guard += 1
                if outer_guard > 8 * (params.max_tokens // self.compact_interval + 2) \
                        + len(prompts) * params.n:
                    raise RuntimeError("sampler scheduling did not converge")

            out = torch.full((len(prompts) * params.n, params.max_tokens), pad_token_id,
                             dtype=torch.long)
            lp_out = torch.zeros(len(prompts) * params.n, params.max_tokens)
            for s in done:
                resp = s.response[: params.max_tokens]
                if resp:
                    out[s.out_index, : len(resp)] = torch.tensor(resp, dtype=torch.long)
                    lps = s.logprobs[: len(resp)]
                    lp_out[s.out_index, : len(lps)] = torch.tensor(lps)
            if return_logprobs:
                return out, lp_out
            return out
        finally:
            if merge_lora:
                unmerge(self.model)
            if was_training:
                self.model.train()
