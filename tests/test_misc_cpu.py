"""Buckets, checkpoint rotation, math verifier, synthetic data, batch algebra."""
import os

import pytest
import torch

from nanorlhf_amd.config import RLHFConfig
from nanorlhf_amd.data import create_batches, hh_shaped_prompts
from nanorlhf_amd.rewards import MathRuleReward
from nanorlhf_amd.rewards.mathcheck import answers_equal, extract_boxed, normalize_answer
from nanorlhf_amd.utils.checkpoint import CheckpointManager


def test_create_batches_budget_invariant():
    lengths = [5, 100, 17, 33, 2, 64, 80, 9]
    budget = 128
    buckets = create_batches(lengths, budget)
    seen = sorted(i for b in buckets for i in b)
    assert seen == list(range(len(lengths)))
    for b in buckets:
        mx = max(lengths[i] for i in b)
        assert mx * len(b) <= budget or len(b) == 1


def test_create_batches_sorted_packing():
    buckets = create_batches([1, 2, 3, 4], 4)
    # sorted by length; [1,2]-> max2*2=4 ok; adding 3 -> 9 > 4
    assert buckets[0] == [0, 1]


def test_batch_algebra_reference_default():
    cfg = RLHFConfig(per_device_train_batch_size=4, gradient_accumulation_steps=8,
                     num_mini_batches=16, total_episodes=1_000_000)
    s = cfg.batch_sizes(world_size=1)
    assert s["local_batch_size"] == 512  # grpo default (grpo_trainer.py:216-247)
    assert s["local_mini_batch_size"] == 32
    s8 = cfg.batch_sizes(world_size=8)
    assert s8["batch_size"] == 4096


def test_extract_boxed():
    assert extract_boxed(r"so the answer is \boxed{42}.") == "42"
    assert extract_boxed(r"\boxed{\frac{1}{2}} and \boxed{x+1}") == "x+1"
    assert extract_boxed("no box here") is None
    assert extract_boxed(r"\boxed{a{b}c}") == "a{b}c"


def test_normalize_and_equal():
    assert normalize_answer(r"\frac{1}{2}") == "((1)/(2))"
    assert answers_equal("42", "42.0")
    assert answers_equal(r"\frac{1}{2}", "0.5")
    assert answers_equal("1,234", "1234")
    assert not answers_equal("41", "42")
    assert answers_equal("x + x", "2x")  # sympy stage


def test_math_rule_reward():
    rw = MathRuleReward(["42", "7"])
    s = rw([r"the answer is \boxed{42}", r"\boxed{8}"])
    assert s.tolist() == [1.0, 0.0]


def test_checkpoint_rotation_and_best(tmp_path):
    cm = CheckpointManager(str(tmp_path), save_total_limit=2,
                           metric_for_best="eval_objective/rlhf_reward_old")
    state = {"w": torch.zeros(2)}
    for step, metric in [(1, 1.0), (2, 5.0), (3, 0.5), (4, 0.1)]:
        cm.save(step, step * 10, state, {"m": 1}, None, None, None,
                {"eval_objective/rlhf_reward_old": metric})
    dirs = sorted(os.listdir(tmp_path))
    # keeps 2 newest + the best; *_old metric at step2 describes checkpoint-1
    assert "checkpoint-4" in dirs and "checkpoint-3" in dirs
    assert os.path.basename(cm.best_checkpoint) == "checkpoint-1"
    loaded = CheckpointManager.load_policy_state(os.path.join(tmp_path, "checkpoint-4"))
    assert "w" in loaded


def test_hh_shaped_prompts_reproducible():
    a = hh_shaped_prompts(5, 1000, seed=3)
    b = hh_shaped_prompts(5, 1000, seed=3)
    assert a == b
    assert all(2 <= t < 1000 for p in a for t in p)


def test_checkpoint_resume_roundtrip(tmp_path):
    """trainer.load_checkpoint restores policy + optimizer + step counters."""
    import torch
    from nanorlhf_amd.algos import reinforce
    from nanorlhf_amd.algos.reinforce import ReinforceConfig
    from nanorlhf_amd.data import hh_shaped_prompts
    from nanorlhf_amd.models import CausalLM
    from nanorlhf_amd.rewards import constant_reward

    def mk(out):
        cfg = ReinforceConfig(model_preset="tiny", dtype="float32", use_lora=True,
                              lora_r=4, lora_alpha=8, per_device_train_batch_size=2,
                              gradient_accumulation_steps=1, num_mini_batches=2,
                              total_episodes=8, response_length=4, temperature=1.0,
                              stop_token_id=1, output_dir=out, save_steps=1,
                              gradient_checkpointing=False, score_token_budget=256)
        torch.manual_seed(0)
        policy = CausalLM.from_preset("tiny")
        ref = CausalLM.from_preset("tiny")
        ref.load_state_dict(policy.state_dict())
        prompts = hh_shaped_prompts(8, 1024, min_len=4, max_len=8)
        return reinforce.make_trainer(cfg, policy, ref,
                                      lambda s: constant_reward(s), prompts)

    t1 = mk(str(tmp_path / "a"))
    t1.train(num_updates=1)
    ck = str(tmp_path / "a" / "checkpoint-1")
    t2 = mk(str(tmp_path / "b"))
    t2.load_checkpoint(ck)
    assert t2.global_step == t1.global_step and t2.episode == t1.episode
    for (n1, p1), (n2, p2) in zip(
            ((n, p) for n, p in t1.policy.named_parameters() if p.requires_grad),
            ((n, p) for n, p in t2.policy.named_parameters() if p.requires_grad)):
        assert n1 == n2 and torch.allclose(p1, p2, atol=1e-7), n1


def test_python_executor_sandbox():
    from nanorlhf_amd.rewards.python_exec import PythonExecutor
    ex = PythonExecutor(timeout_s=3.0)
    r = ex.run("answer = 6*7\nprint('hi')")
    assert r["ok"] and r["answer"] == 42 and "hi" in r["stdout"]
    r2 = ex.run("while True: pass")
    assert not r2["ok"] and r2["error"] == "timeout"
    r3 = ex.run("raise ValueError('x')")
    assert not r3["ok"]


def test_early_stopping_callback():
    from nanorlhf_amd.utils.callbacks import EarlyStoppingCallback
    cb = EarlyStoppingCallback(metric="m", patience=2, greater_is_better=True)
    assert not cb.on_update_end(None, {"m": 1.0})
    assert not cb.on_update_end(None, {"m": 0.9})
    assert cb.on_update_end(None, {"m": 0.8})  # second bad step -> stop


def test_disable_dropout():
    import torch
    from nanorlhf_amd.algos.functional import disable_dropout_in_model
    m = torch.nn.Sequential(torch.nn.Linear(2, 2), torch.nn.Dropout(0.5))
    disable_dropout_in_model(m)
    assert m[1].p == 0.0


def test_math_aliases_and_extraction():
    from nanorlhf_amd.rewards.mathcheck import (extract_math_answer, is_correct,
                                                is_equiv, latex_answer_check,
                                                math_equal)
    assert extract_math_answer(r"thus \boxed{12}") == "12"
    assert extract_math_answer("the result is 3.5 meters") == "3.5"
    assert extract_math_answer("no numbers") is None
    for fn in (is_correct, is_equiv, latex_answer_check, math_equal):
        assert fn("42", "42.0")
        assert not fn("41", "42")


def test_mathcheck_pathological_timeout_fast():
    """sympy bombs must be cut off by the subprocess timeout quickly."""
    import time
    from nanorlhf_amd.rewards.mathcheck import answers_equal
    t0 = time.time()
    out = answers_equal("x**x**x**x**99999 + y", "z", 0.3)
    assert out is False
    assert time.time() - t0 < 5.0


def test_a_changed_header_compiles_every_source_again(tmp_path, monkeypatch):
    """Sources are compiled again when their command changes; headers are not tracked."""
    import runpy
    import shutil
    from types import SimpleNamespace
    import setuptools
    import torch.utils.cpp_extension as cpp
    seen = []
    monkeypatch.setattr(cpp, "CUDAExtension", lambda **k: SimpleNamespace(**k))
    monkeypatch.setattr(setuptools, "setup", lambda **k: seen.append(
        [e.extra_compile_args for e in k["ext_modules"]]))
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    shutil.copy(os.path.join(root, "setup.py"), tmp_path)
    csrc = tmp_path / "nanorlhf_amd" / "csrc"
    csrc.mkdir(parents=True)
    for text in ("one", "one", "two"):
        (csrc / "common.h").write_text(text)
        runpy.run_path(str(tmp_path / "setup.py"))
    assert seen[0] == seen[1]
    for before, after in zip(seen[1], seen[2]):
        assert all(before[kind] != after[kind] for kind in ("cxx", "nvcc"))
