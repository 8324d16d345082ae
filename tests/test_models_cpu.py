"""CPU model tests: shapes, packing, GQA, scalar heads, LoRA."""
import pytest
import torch

from nanorlhf_amd.models import (AttnContext, CausalLM, LoraConfig, ScalarHeadModel,
                                 apply_lora, get_config, pack_sequences)
from nanorlhf_amd.models.lora import LoRALinear, merge_for_rollout, unmerge
from nanorlhf_amd.ops import build_rope_cache, rope_apply


def _fwd(model, seqs):
    ids, cu, mx, pos = pack_sequences(seqs)
    return model(ids, CausalLM.train_ctx(cu, mx, pos))


def test_packed_forward_matches_per_sequence():
    torch.manual_seed(0)
    m = CausalLM.from_preset("tiny").eval()
    seqs = [torch.randint(2, 1000, (n,)) for n in (9, 5, 13)]
    h_all = _fwd(m, seqs)
    off = 0
    for s in seqs:
        h_one = _fwd(m, [s])
        assert torch.allclose(h_all[off:off + len(s)], h_one, atol=1e-4)
        off += len(s)


def test_causal_dependence():
    """Changing a later token must not change earlier hidden states."""
    torch.manual_seed(0)
    m = CausalLM.from_preset("tiny").eval()
    s = torch.randint(2, 1000, (10,))
    h1 = _fwd(m, [s])
    s2 = s.clone()
    s2[-1] = (s2[-1] + 1) % 1000
    h2 = _fwd(m, [s2])
    assert torch.allclose(h1[:-1], h2[:-1], atol=1e-5)
    assert not torch.allclose(h1[-1], h2[-1], atol=1e-5)


def test_rope_orthogonal_and_inverse():
    table = build_rope_cache(32, 64, theta=1e4)
    x = torch.randn(5, 2, 32)
    pos = torch.arange(5)
    y = rope_apply(x, table, pos)
    # norms preserved (rotation)
    assert torch.allclose(x.norm(dim=-1), y.norm(dim=-1), atol=1e-4)
    # position 0 is identity
    assert torch.allclose(y[0], x[0], atol=1e-6)


def test_scalar_head_sequence_scores():
    torch.manual_seed(0)
    rm = ScalarHeadModel.from_preset("rm-tiny").eval()
    seqs = [torch.randint(2, 1000, (n,)) for n in (6, 11)]
    ids, cu, mx, _ = pack_sequences(seqs)
    s = rm.sequence_scores(ids, cu, mx)
    assert s.shape == (2,)
    v = rm.token_values(ids, cu, mx)
    assert v.shape == (ids.numel(),)


def test_bidirectional_rm_sees_future():
    torch.manual_seed(0)
    rm = ScalarHeadModel.from_preset("rm-tiny").eval()
    assert rm.cfg.bidirectional
    s = torch.randint(2, 1000, (8,))
    ids, cu, mx, _ = pack_sequences([s])
    v1 = rm.token_values.__wrapped__ if hasattr(rm.token_values, "__wrapped__") else None
    # change LAST token; FIRST token's score should change under bidirectional attn
    from nanorlhf_amd.models.qwen2 import AttnContext, make_positions
    ctx = AttnContext(mode="train", positions=make_positions(cu), cu_seqlens=cu, max_seqlen=mx)
    out1 = rm(ids, ctx)
    s2 = s.clone(); s2[-1] = (s2[-1] + 1) % 1000
    ids2, cu2, mx2, _ = pack_sequences([s2])
    ctx2 = AttnContext(mode="train", positions=make_positions(cu2), cu_seqlens=cu2, max_seqlen=mx2)
    out2 = rm(ids2, ctx2)
    assert not torch.allclose(out1[0], out2[0], atol=1e-6)


def test_lora_apply_merge_unmerge():
    torch.manual_seed(0)
    m = CausalLM.from_preset("tiny")
    apply_lora(m, LoraConfig(r=4, alpha=8))
    trainable = [n for n, p in m.named_parameters() if p.requires_grad]
    assert any("lora_A" in n for n in trainable)
    assert any("embed_tokens" in n for n in trainable)
    assert not any(n.endswith("base.weight") for n in trainable)
    s = torch.randint(2, 1000, (7,))
    m.eval()
    h0 = _fwd(m, [s])
    # B is zero-init → merged == unmerged at init
    merge_for_rollout(m)
    h1 = _fwd(m, [s])
    unmerge(m)
    assert torch.allclose(h0, h1, atol=1e-5)
    # after perturbing B, lora path changes output
    for mod in m.modules():
        if isinstance(mod, LoRALinear):
            torch.nn.init.normal_(mod.lora_B, std=0.1)
    h2 = _fwd(m, [s])
    assert not torch.allclose(h0, h2, atol=1e-4)
    # merged path equals unmerged compute path
    merge_for_rollout(m)
    h3 = _fwd(m, [s])
    assert torch.allclose(h2, h3, atol=1e-4)
    unmerge(m)


def test_tied_and_untied_lm_head():
    tied = CausalLM(get_config("tiny", tie_word_embeddings=True))
    untied = CausalLM(get_config("tiny", tie_word_embeddings=False))
    assert tied.lm_head is None
    assert tied.lm_head_weight.data_ptr() == tied.model.embed_tokens.weight.data_ptr()
    assert untied.lm_head is not None


@pytest.mark.parametrize("preset", ["tiny", "gonurax-tiny", "bedalorn-tiny"])
def test_model_built_inside_a_device_context_is_all_there(preset):
    """Every tensor of a model built under torch.device(...) is on that device:
    a table left on the host would be a host pointer in a kernel."""
    from nanorlhf_amd.models import build_model, get_config
    with torch.device("meta"):
        m = build_model(get_config(preset))
    assert {t.device.type for t in [*m.parameters(), *m.buffers()]} == {"meta"}


def test_rope_table_follows_the_default_device():
    want = build_rope_cache(32, 64)
    assert want.device.type == "cpu" and want.dtype == torch.float32
    with torch.device("meta"):
        assert build_rope_cache(32, 64).device.type == "meta"
        assert torch.equal(build_rope_cache(32, 64, device="cpu"), want)


@pytest.fixture
def in_parts(monkeypatch):
    """Projections of float32 rows return two parts of their depth where they may."""
    from nanorlhf_amd import ops

    def linear_parts(x, w, bias=None):
        half = w.shape[1] // 2
        return torch.stack([x[:, :half] @ w[:, :half].T, x[:, half:] @ w[:, half:].T])

    monkeypatch.setattr(ops, "linear_parts", linear_parts)


@pytest.mark.parametrize("name", ["Attention", "MLP", "Block"])
def test_replaced_forwards_of_a_class_are_called_as_they_were(monkeypatch, in_parts, name):
    """What a program puts in a class's place knows nothing of parts and gets none."""
    from nanorlhf_amd.models import qwen2
    m, s = CausalLM.from_preset("tiny").eval(), torch.arange(2, 9)
    cls, shapes = getattr(qwen2, name), []
    own = cls.forward

    def forward(self, *args):
        shapes.extend(tuple(a.shape) for a in args[:2 if name == "Block" else 1] if a is not None)
        out = own(self, *args)
        shapes.extend(tuple(t.shape) for t in (out if isinstance(out, tuple) else (out,)))
        return out

    with torch.no_grad():
        want = _fwd(m, [s])
        monkeypatch.setattr(cls, "forward", forward)
        got = _fwd(m, [s])
    assert set(shapes) == {(7, m.cfg.hidden_size)}
    assert torch.allclose(got, want, atol=1e-5)


@pytest.mark.parametrize("how", ["pre-hook", "hook", "subclass", "instance", "wrapped"])
def test_a_layer_that_is_not_plain_is_given_sums_and_no_parts(monkeypatch, in_parts, how):
    from nanorlhf_amd import ops
    from nanorlhf_amd.models.qwen2 import Block
    m, s = CausalLM.from_preset("tiny", num_layers=3).eval(), torch.arange(2, 9)
    layers, normed, seen = m.model.layers, [], []
    plain, norm = layers[1], ops.add_parts_rms_norm
    monkeypatch.setattr(ops, "add_parts_rms_norm",
                        lambda x, *args: (normed.append(x.dim()), norm(x, *args))[1])
    with torch.no_grad():
        want = _fwd(m, [s])
    assert normed == [2] + [3] * 6          # but the embedding all of them are parts

    class Sub(Block):
        def forward(self, delta, res, *args):
            seen.append(delta.shape)
            return super().forward(delta, res, *args)

    class Wrapped(torch.nn.Module):
        def forward(self, delta, res, *args):
            seen.append(delta.shape)
            return plain(delta, res, *args)

    if how == "pre-hook":
        plain.register_forward_pre_hook(lambda mod, args: seen.append(args[0].shape))
    elif how == "hook":
        plain.register_forward_hook(lambda mod, args, out: seen.append(args[0].shape))
    elif how == "subclass":
        plain.__class__ = Sub
    elif how == "wrapped":
        layers[1] = Wrapped()
    else:
        own = plain.forward
        plain.forward = lambda delta, *args: (seen.append(delta.shape), own(delta, *args))[1]
    with torch.no_grad():
        got = _fwd(m, [s])
    assert seen == [(7, m.cfg.hidden_size)]
    assert torch.allclose(got, want, atol=1e-5)
