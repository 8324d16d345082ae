"""HIP kernel dispatch layer.

Every hot op has two paths:
  * GPU (``tensor.is_cuda``): the hand-written gfx950 HIP kernel from the
    in-tree extensions ``nanorlhf_amd/_C.so`` (training, scoring, sampling)
    and ``nanorlhf_amd/_serve.so`` (paged cache, attention over it, linear
    attention, residual-stream kernels); the linears without gradients are
    in both.  If an extension is missing on a machine with a GPU this raises
    loudly — there is NO silent eager fallback on GPU.
  * CPU: a plain-PyTorch fp32 reference used by the CPU test suite and as
    the numerics oracle for the kernels.
"""
from __future__ import annotations

import importlib

import torch  # noqa: F401  (must load before the extensions: provides libc10)

_LOADED: dict = {}


def _load(name: str):
    if name not in _LOADED:
        try:
            _LOADED[name] = (importlib.import_module(f"nanorlhf_amd.{name}"), None)
        except Exception as e:  # noqa: BLE001
            _LOADED[name] = (None, e)
    return _LOADED[name]


def _require(name: str):
    m, err = _load(name)
    if m is None:
        raise RuntimeError(
            f"nanorlhf_amd.{name} HIP extension is not built/importable but a GPU op "
            "was requested. Build it in-tree with `python setup.py build_ext "
            f"--inplace` (PYTORCH_ROCM_ARCH=gfx950). Original error: {err!r}"
        )
    return m


def ext():
    """The training/sampling extension; raises loudly if unavailable."""
    return _require("_C")


def serve_ext():
    """The serving extension; raises loudly if unavailable."""
    return _require("_serve")


def linear_ext():
    """The linears without gradients, which scoring and serving both run: either
    extension has them; raises loudly if neither is available."""
    return _require("_serve" if _load("_serve")[0] is not None else "_C")


def ext_available() -> bool:
    return all(_load(n)[0] is not None for n in ("_C", "_serve"))


from .rmsnorm import (add_parts_rms_norm, add_rms_norm, gated_norm,  # noqa: E402,F401
                      residual_group_norm, rms_norm)
from .rope import Rotation, build_rope_cache, qkv_rope, rope_apply  # noqa: E402,F401
from .linear import linear, linear_parts, sum_parts  # noqa: E402,F401
from .swiglu import (gelu_glu, glu_fuses, linear_gelu_glu, linear_swiglu,  # noqa: E402,F401
                     relu_squared_, swiglu)
from .attention import flash_attn_varlen  # noqa: E402,F401
from .logprob import token_logprob_entropy  # noqa: E402,F401
from .adamw import FusedAdamW  # noqa: E402,F401
from .sampling import sample_tokens  # noqa: E402,F401
from .kvcache import (kv_append, paged_attn, paged_attn_decode,  # noqa: E402,F401
                      pad_head_dim, qkv_rope_append, rotary_qkv)
from .latent import latent_append, latent_attn, pad_latent  # noqa: E402,F401
from .moe import group_linear, moe_experts, moe_route, stacked_linear  # noqa: E402,F401
from .wkv import token_shift, wkv, wkv_decay  # noqa: E402,F401
from .linear_attn import DecayTable, linear_attn_chunked, linear_attn_decode  # noqa: E402,F401
