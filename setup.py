"""Build the in-tree gfx950 HIP extensions:

    PYTORCH_ROCM_ARCH=gfx950 python setup.py build_ext --inplace

  nanorlhf_amd/_C      training, scoring and sampling kernels
  nanorlhf_amd/_serve  paged cache, attention over it, linear attention,
                       mixture of experts and residual-stream kernels (all a
                       model forward needs when it is served)

NANORLHF_EXT=_serve builds just that one.  The .so files are git-ignored."""
import hashlib
import os

from setuptools import setup

os.environ.setdefault("PYTORCH_ROCM_ARCH", "gfx950")

from torch.utils.cpp_extension import BuildExtension, CUDAExtension  # noqa: E402

ROOT = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(ROOT, "nanorlhf_amd", "csrc")

LINEAR = ["glu.hip", "linear_rows.hip"]     # both have them, so that each serves alone
EXTENSIONS = {
    "_C": ["bindings.cpp", "elementwise.hip", "logprob.hip", "adamw.hip",
           "sampling.hip", "attention.hip", "masked.hip", "lora.hip",
           "lora_grad.hip", *LINEAR],
    "_serve": ["serve_bindings.cpp", "kvcache.hip", "paged_attention.hip",
               "linear_attn.hip", "stream.hip", "wkv.hip", "latent_attn.hip", "moe.hip",
               *LINEAR],
}



def headers():
    """What the headers say, as a number: the sources' dependences on them are not tracked, but
    a changed command compiles a source again."""
    digest = hashlib.sha256()
    for name in sorted(f for f in os.listdir(CSRC) if f.endswith(".h")):
        with open(os.path.join(CSRC, name), "rb") as f:
            digest.update(name.encode() + b"\0" + f.read())
    return f"-DNANORLHF_HEADERS=0x{digest.hexdigest()[:16]}"


wanted = [n for n in os.environ.get("NANORLHF_EXT", "").split(",") if n] or list(EXTENSIONS)

setup(
    name="nanorlhf_amd_C",
    ext_modules=[
        CUDAExtension(
            name=f"nanorlhf_amd.{name}",
            sources=[os.path.join(CSRC, f) for f in EXTENSIONS[name]],
            extra_compile_args={
                "cxx": ["-O3", "-std=c++17", headers()],
                # no packed fp32 VALU forms: some give wrong results on this part
                "nvcc": ["-O3", "-std=c++17", "--offload-arch=gfx950", headers(),
                         "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"],
            },
        )
        for name in wanted
    ],
    cmdclass={"build_ext": BuildExtension},
)
