"""Pure algorithm math shared by every trainer.

Each function is a semantics-preserving re-implementation of the math the
reference inlines inside its six ``<algo>_trainer.py`` ``train()`` bodies,
whose call sites each function cites.  Everything here is device-agnostic
torch; the hot token-level pieces have HIP-fused twins in ``nanorlhf_amd.ops``
which these functions dispatch to on GPU where it pays.
"""
from __future__ import annotations

import torch

# Padding sentinel for logprobs of non-response positions.
# Reference quirk preserved: GRPO/grpo_trainer.py:81 (INVALID_LOGPROB = 1.0).
INVALID_LOGPROB = 1.0


def disable_dropout_in_model(model: torch.nn.Module) -> torch.nn.Module:
    """Set every Dropout's p to 0 (trl helper imported at
    grpo_trainer.py:58-71; our models only carry LoRA dropout)."""
    for m in model.modules():
        if isinstance(m, torch.nn.Dropout):
            m.p = 0.0
    return model


def masked_mean(values: torch.Tensor, mask: torch.Tensor, axis=None) -> torch.Tensor:
    """Mean of `values` over positions where mask==1.

    Re-implements the trl helper imported at GRPO/grpo_trainer.py:54.
    """
    if axis is not None:
        return (values * mask).sum(axis=axis) / mask.sum(axis=axis)
    return (values * mask).sum() / mask.sum()


def masked_var(values: torch.Tensor, mask: torch.Tensor, unbiased: bool = True) -> torch.Tensor:
    mean = masked_mean(values, mask)
    centered = values - mean
    var = masked_mean(centered**2, mask)
    if unbiased:
        n = mask.sum()
        var = var * n / torch.clamp(n - 1, min=1)
    return var


def masked_whiten(values: torch.Tensor, mask: torch.Tensor, shift_mean: bool = True) -> torch.Tensor:
    """Whiten `values` using masked moments (trl semantics, grpo_trainer.py:607,619).

    GPU: fused HIP masked-moments + apply kernels (no grad flows through the
    whitening of advantages); CPU: plain torch reference."""
    if values.is_cuda and not values.requires_grad and values.dtype == torch.float32:
        from .. import ops as _ops
        vc = values.contiguous()
        mc = mask.contiguous().float()
        (partials,) = _ops.ext().masked_moments(vc.view(-1), mc.view(-1))
        sums = partials.sum(0)  # [sum, sumsq, count]
        cnt = sums[2].clamp(min=1.0)
        mean = sums[0] / cnt
        var = (sums[1] / cnt - mean * mean) * cnt / (cnt - 1.0).clamp(min=1.0)
        invstd = torch.rsqrt(var + 1e-8)
        # trl semantics: shift_mean=True -> zero-centered; False -> mean kept.
        shift = torch.zeros_like(mean) if shift_mean else mean
        out = _ops.ext().whiten_apply(vc.view(-1), float(mean), float(invstd),
                                      float(shift))
        return out.view_as(values)
    mean = masked_mean(values, mask)
    var = masked_var(values, mask)
    whitened = (values - mean) * torch.rsqrt(var + 1e-8)
    if not shift_mean:
        whitened = whitened + mean
    return whitened


def first_true_indices(bools: torch.Tensor, dtype=torch.long) -> torch.Tensor:
    """Index of the first True along dim=-1; length of the row if none.

    trl helper used for EOS detection (grpo_trainer.py:58-71 imports).
    """
    row_len = bools.size(-1)
    zero_or_index = row_len * (~bools).type(dtype) + torch.arange(row_len, dtype=dtype, device=bools.device)
    return torch.min(zero_or_index, dim=-1).values


def truncate_response(stop_token_id: int, pad_token_id: int, responses: torch.Tensor) -> torch.Tensor:
    """Replace everything after the first stop token with pad (grpo_trainer.py:560-562)."""
    trunc_idxs = first_true_indices(responses == stop_token_id).unsqueeze(-1)
    idxs = torch.arange(responses.shape[1], device=responses.device).repeat(responses.shape[0], 1)
    return torch.masked_fill(responses, idxs > trunc_idxs, pad_token_id)


def exact_div(a: int, b: int, custom_error_message: str = "") -> int:
    q = a // b
    if a != q * b:
        raise ValueError(f"{custom_error_message}, inexact division: {a} / {b} = {a / b}")
    return q


# ---------------------------------------------------------------------------
# Advantage constructions (one per algorithm)
# ---------------------------------------------------------------------------

def grpo_group_advantage(scores: torch.Tensor, n: int) -> torch.Tensor:
    """Group-relative advantage: per prompt-group of n samples, (x-mean)/std.

    Semantics of GRPO/grpo_trainer.py:502-520 including the std nan guard
    (nan→0 when a group is degenerate, :508-512).

    scores: [B*n] flat, grouped so that rows [i*n:(i+1)*n] share a prompt.
    Returns [B*n].
    """
    g = scores.view(-1, n)
    mean = g.mean(dim=1, keepdim=True)
    std = g.std(dim=1, keepdim=True)
    adv = (g - mean) / std
    adv = torch.nan_to_num(adv, nan=0.0, posinf=0.0, neginf=0.0)
    return adv.reshape(-1)


def random_keep_one_per_group(batch: int, n: int, generator: torch.Generator | None = None,
                              device="cpu") -> torch.Tensor:
    """Indices keeping 1 random sample of each n-group (grpo_trainer.py:513-520,
    rloo_trainer.py:603-613 — "abandon some examples to save time")."""
    offsets = torch.randint(0, n, (batch,), generator=generator, device=device)
    return torch.arange(batch, device=device) * n + offsets


def rloo_baseline_advantage(rlhf_reward: torch.Tensor, n: int) -> torch.Tensor:
    """Leave-one-out baseline (RLOO/rloo_trainer.py:597-599).

    rlhf_reward: [B*n] sequence-level (KL-shaped) rewards, grouped per prompt.
    adv_i = r_i - mean(r_{j != i}).
    """
    g = rlhf_reward.view(-1, n)
    baseline = (g.sum(dim=1, keepdim=True) - g) / max(n - 1, 1)
    return (g - baseline).reshape(-1)


def remax_advantage(scores_sampled: torch.Tensor, scores_greedy: torch.Tensor) -> torch.Tensor:
    """ReMax: sampled reward minus greedy-baseline reward (remax_trainer.py:506-513)."""
    return scores_sampled - scores_greedy


def reward_to_go(rewards: torch.Tensor, gamma: float = 1.0) -> torch.Tensor:
    """Undiscounted (gamma=1) or discounted reward-to-go scan over time.

    rewards: [B, T].  adv[:, t] = rewards[:, t] + gamma * adv[:, t+1].
    GRPO variant (gamma=1): grpo_trainer.py:611-620; REINFORCE variant with
    config gamma: reinforce_trainer.py:583-587.

    Implemented as a vectorized reverse scan (gamma=1 → reversed cumsum) —
    the reference's per-timestep Python loop is kept only as the test oracle.
    """
    if gamma == 1.0:
        return torch.flip(torch.cumsum(torch.flip(rewards, dims=[1]), dim=1), dims=[1])
    T = rewards.size(1)
    out = torch.empty_like(rewards)
    acc = torch.zeros_like(rewards[:, 0])
    for t in range(T - 1, -1, -1):
        acc = rewards[:, t] + gamma * acc
        out[:, t] = acc
    return out


def gae(rewards: torch.Tensor, values: torch.Tensor, gamma: float, lam: float) -> tuple[torch.Tensor, torch.Tensor]:
    """Generalized advantage estimation (PPO/ppo_trainer.py:688-697).

    rewards, values: [B, T].  Returns (advantages, returns) with
    returns = advantages + values (:697).  Terminal value beyond T is 0.
    """
    T = rewards.size(1)
    lastgaelam = torch.zeros_like(rewards[:, 0])
    adv_rev = []
    for t in range(T - 1, -1, -1):
        nextvalues = values[:, t + 1] if t < T - 1 else torch.zeros_like(values[:, t])
        delta = rewards[:, t] + gamma * nextvalues - values[:, t]
        lastgaelam = delta + gamma * lam * lastgaelam
        adv_rev.append(lastgaelam)
    advantages = torch.stack(adv_rev[::-1], dim=1)
    returns = advantages + values
    return advantages, returns


def sparse_reward_at_eos(scores: torch.Tensor, response_mask: torch.Tensor,
                         eos_indices: torch.Tensor) -> torch.Tensor:
    """Scatter the sequence score at the EOS position of each response
    (grpo_trainer.py:598-603): rewards[b, eos_idx[b]] = scores[b], 0 elsewhere.
    """
    rewards = torch.zeros_like(response_mask, dtype=scores.dtype)
    rows = torch.arange(scores.size(0), device=scores.device)
    idx = eos_indices.clamp(max=response_mask.size(1) - 1)
    rewards[rows, idx] = scores
    return rewards


def kl_shaped_rewards(scores: torch.Tensor, logprobs: torch.Tensor, ref_logprobs: torch.Tensor,
                      response_mask: torch.Tensor, eos_indices: torch.Tensor,
                      kl_coef: float) -> torch.Tensor:
    """Per-token reward stream = -kl_coef * (logp - ref_logp), plus the
    sequence score added at the EOS index (PPO/ppo_trainer.py:672-674,
    RLOO/rloo_trainer.py:571-573, reinforce_trainer.py:568-570).
    """
    kl = logprobs - ref_logprobs
    rewards = -kl_coef * kl
    rows = torch.arange(scores.size(0), device=scores.device)
    idx = eos_indices.clamp(max=response_mask.size(1) - 1)
    rewards[rows, idx] = rewards[rows, idx] + scores
    return rewards * response_mask


# ---------------------------------------------------------------------------
# Losses
# ---------------------------------------------------------------------------

def ppo_clip_token_loss(new_logprobs: torch.Tensor, old_logprobs: torch.Tensor,
                        advantages: torch.Tensor, mask: torch.Tensor,
                        cliprange: float) -> tuple[torch.Tensor, dict]:
    """Token-level PPO clipped surrogate (grpo_trainer.py:652-690 and the
    ReMax/REINFORCE twins).  Returns (loss, stats)."""
    logprobs_diff = new_logprobs - old_logprobs
    ratio = torch.exp(logprobs_diff)
    pg_losses = -advantages * ratio
    pg_losses2 = -advantages * torch.clamp(ratio, 1.0 - cliprange, 1.0 + cliprange)
    pg_loss_max = torch.max(pg_losses, pg_losses2)
    pg_loss = masked_mean(pg_loss_max, mask)
    with torch.no_grad():
        pg_clipfrac = masked_mean((pg_losses2 > pg_losses).float(), mask)
        approxkl = 0.5 * masked_mean(logprobs_diff**2, mask)
    return pg_loss, {"pg_clipfrac": pg_clipfrac, "approxkl": approxkl, "ratio": ratio.detach()}


def rloo_sequence_loss(new_logprobs: torch.Tensor, old_logprobs: torch.Tensor,
                       advantages_seq: torch.Tensor, mask: torch.Tensor,
                       cliprange: float) -> tuple[torch.Tensor, dict]:
    """Sequence-level ratio PPO-clip (RLOO/rloo_trainer.py:660-669):
    ratio = exp(sum_t new - sum_t old), one advantage per sequence."""
    new_sum = (new_logprobs * mask).sum(1)
    old_sum = (old_logprobs * mask).sum(1)
    logprobs_diff = new_sum - old_sum
    ratio = torch.exp(logprobs_diff)
    pg_losses = -advantages_seq * ratio
    pg_losses2 = -advantages_seq * torch.clamp(ratio, 1.0 - cliprange, 1.0 + cliprange)
    pg_loss_max = torch.max(pg_losses, pg_losses2)
    pg_loss = pg_loss_max.mean()
    with torch.no_grad():
        pg_clipfrac = (pg_losses2 > pg_losses).float().mean()
        approxkl = 0.5 * (logprobs_diff**2).mean()
    return pg_loss, {"pg_clipfrac": pg_clipfrac, "approxkl": approxkl, "ratio": ratio.detach()}


def raft_nll_loss(new_logprobs: torch.Tensor, mask: torch.Tensor) -> torch.Tensor:
    """Best-of-K SFT loss: plain NLL over the selected responses
    (RAFT/raft_trainer.py:636): -sum_t logp, mean over batch."""
    return -(new_logprobs * mask).sum(1).mean()


def k3_kl_penalty(new_logprobs: torch.Tensor, ref_logprobs: torch.Tensor,
                  kl_coef: float) -> torch.Tensor:
    """k3 KL estimator penalty added to the GRPO loss (grpo_trainer.py:667-670):
    kl_coef * (e^{-kl} + kl - 1), kl = new - ref.  Non-negative, unbiased-ish."""
    kl = new_logprobs - ref_logprobs
    return kl_coef * (torch.exp(-kl) + kl - 1.0)


def value_clip_loss(vpred: torch.Tensor, old_values: torch.Tensor, returns: torch.Tensor,
                    mask: torch.Tensor, cliprange_value: float) -> tuple[torch.Tensor, torch.Tensor]:
    """Clipped value MSE (PPO/ppo_trainer.py:742-749). Returns (vf_loss, clipfrac)."""
    vpredclipped = torch.clamp(vpred, old_values - cliprange_value, old_values + cliprange_value)
    vf_losses1 = (vpred - returns) ** 2
    vf_losses2 = (vpredclipped - returns) ** 2
    vf_loss_max = torch.max(vf_losses1, vf_losses2)
    vf_loss = 0.5 * masked_mean(vf_loss_max, mask)
    vf_clipfrac = masked_mean((vf_losses2 > vf_losses1).float(), mask)
    return vf_loss, vf_clipfrac


def entropy_from_logits(logits: torch.Tensor) -> torch.Tensor:
    """H = logsumexp(logits) - sum softmax*logits (grpo_trainer.py:678-679).

    CPU/test reference for the fused HIP logprob+entropy kernel."""
    pd = torch.nn.functional.softmax(logits, dim=-1)
    return torch.logsumexp(logits, dim=-1) - torch.sum(pd * logits, dim=-1)


def missing_eos_penalty(scores: torch.Tensor, responses: torch.Tensor, eos_token_id: int,
                        penalty: float) -> torch.Tensor:
    """Subtract `penalty` from sequences that never emitted EOS
    (grpo_trainer.py:584-586)."""
    contains_eos = (responses == eos_token_id).any(dim=1)
    return torch.where(contains_eos, scores, scores - penalty)
