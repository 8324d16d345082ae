"""GPU kernels at the sizes where a tile, a split or a vector load ends: against
the plain references in 32 or 64 bits."""
import pytest
import torch

from nanorlhf_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


def rnd(*shape, seed, scale=1.0, dtype=torch.bfloat16):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return (torch.randn(*shape, generator=g, device=DEV) * scale).to(dtype)


def rel(a, b):
    a, b = a.double(), b.double()
    return float((a - b).norm() / (b.norm() + 1e-30))


# P and dS are rounded to bf16 on the way into the second products and the
# results once more, each 2^-9 at most and 0.0011 in the root mean square; dS also
# carries the difference dP - D of numbers about twice its size.
FA_REL = 0.01


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("hq,hkv,d", [(12, 2, 128), (7, 1, 64), (4, 4, 64), (4, 2, 32)])
@pytest.mark.parametrize("lens", [[1, 31, 32, 33, 63, 64, 65, 127, 128, 129, 257],
                                  [1 + i % 21 for i in range(800)]])    # parts: several, one
def test_flash_attention_tile_edges(lens, hq, hkv, d, causal):
    from nanorlhf_amd.ops.attention import _sdpa_ref_autograd
    T = sum(lens)
    cu = torch.tensor([0] + lens, device=DEV).cumsum(0).int()
    q, k, v = rnd(T, hq, d, seed=1, scale=2.0), rnd(T, hkv, d, seed=2), rnd(T, hkv, d, seed=3)
    do = rnd(T, hq, d, seed=4)
    leaves = [t.clone().requires_grad_(True) for t in (q, k, v)]
    o = ops.flash_attn_varlen(*leaves, cu, max(lens), causal=causal)
    o.backward(do)
    exact = [t.float().requires_grad_(True) for t in (q, k, v)]
    want = _sdpa_ref_autograd(*exact, cu.cpu(), d ** -0.5, causal=causal)
    want.backward(do.float())
    assert rel(o, want) < FA_REL
    for got, ref in zip(leaves, exact):
        assert rel(got.grad, ref.grad) < FA_REL


def test_flash_attention_negative_and_zero_scale():
    lens = [70, 130]
    cu = torch.tensor([0] + lens, device=DEV).cumsum(0).int()
    q, k, v = rnd(200, 4, 64, seed=1), rnd(200, 2, 64, seed=2), rnd(200, 2, 64, seed=3)
    from nanorlhf_amd.ops.attention import _sdpa_ref
    for scale in (-0.2, 0.0):
        o = ops.flash_attn_varlen(q, k, v, cu, max(lens), scale=scale)
        assert rel(o, _sdpa_ref(q.float(), k.float(), v.float(), cu.cpu(), scale)) < FA_REL
