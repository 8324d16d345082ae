// Gated feed-forward's first half in one product: out = act(x Wg^T) * (x Wu^T),
// the activation in 32-bit before the only rounding.  Two products (or one of both
// widths) and a pass over their results took three trips through memory for what
// is written once here.
//
// The tile is gemm_big.h's, and so are its bounds.  16320 x 8960 x 1536: 0.66 ms
// (1360 TFLOP/s), where the library's product of both widths takes 0.66 and the pass 0.16.
#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>

#include "common.h"
#include "checks.h"
#include "gemm_big.h"

// x [M, K], gate and up [N, K] (rows contiguous), out [M, >= N] of any row stride;
// act 0: silu, 1: gelu_tanh
void glu_linear(torch::Tensor x, torch::Tensor gate, torch::Tensor up, torch::Tensor out,
                long act) {
  on_gpu({x, gate, up, out});
  for (const auto& t : {x, gate, up, out})
    TORCH_CHECK(t.dim() == 2 && t.scalar_type() == torch::kBFloat16 && t.stride(1) == 1,
                "glu_linear: bf16 matrices with contiguous rows");
  const long M = x.size(0), K = x.size(1), N = gate.size(0);
  TORCH_CHECK(x.is_contiguous() && gate.is_contiguous() && up.is_contiguous() &&
              gate.size(1) == K && up.sizes() == gate.sizes() && out.size(0) == M &&
              out.size(1) == N, "glu_linear: shapes");
  TORCH_CHECK(K % 64 == 0 && K > 0, "glu_linear: depth must be a multiple of 64");
  for (const auto& t : {x, gate, up})
    TORCH_CHECK((uintptr_t)t.data_ptr() % 16 == 0, "glu_linear: operands on 16 bytes");
  TORCH_CHECK(act == 0 || act == 1, "glu_linear: activation");
  if (M == 0 || N == 0) return;
  const long gm = (M + BIG - 1) / BIG, gn = (N + BIG / 2 - 1) / (BIG / 2);
  TORCH_CHECK(gm * gn < (1L << 31) && K < (1L << 22), "glu_linear: too large");
  const long ldo = out.stride(0);
  const bool vec = N % 4 == 0 && ldo % 4 == 0 && (uintptr_t)out.data_ptr() % 8 == 0;
  Big p{};
  p.x = (const short*)x.data_ptr();
  p.w = (const short*)gate.data_ptr();
  p.w2 = (const short*)up.data_ptr();
  p.y = (short*)out.data_ptr();
  p.ldy = ldo;
  p.M = M;
  p.N = N;
  p.K = K;
#define LAUNCH(VEC, ACT) launch_big<false, false, VEC, ACT>(p)
  if (act == 0) { if (vec) LAUNCH(true, SILU_GLU); else LAUNCH(false, SILU_GLU); }
  else { if (vec) LAUNCH(true, GELU_GLU); else LAUNCH(false, GELU_GLU); }
#undef LAUNCH
  HIP_CHECK_LAST();
}
