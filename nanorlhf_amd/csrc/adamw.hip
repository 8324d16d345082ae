// Fused AdamW step: one pass over (p, g, m, v) with fp32 state, decoupled
// weight decay and bias correction; bf16 or fp32 params.
//
// Up to 64 tensors per launch, their pointers in the kernel's arguments: the
// hundreds of small adapters of a LoRA model cost a launch each otherwise.
// Bound by memory: 22 bytes per bf16 parameter.
#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>

#include "common.h"

constexpr int AT_ONCE = 64, PER_BLOCK = 256 * 8 * 2;     // tensors, elements

struct AdamTensors {
  void* p[AT_ONCE];
  const void* g[AT_ONCE];
  float* m[AT_ONCE];
  float* v[AT_ONCE];
  long n[AT_ONCE];
  int first[AT_ONCE + 1];    // first workgroup of each tensor
  unsigned long long vec;    // bit per tensor: 16-byte accesses
};

struct AdamRates { float lr, b1, b2, eps, wd, bc1, bc2; };

DEVINL float adam_one(float p, float g, float& m, float& v, const AdamRates& r) {
  m = r.b1 * m + (1.f - r.b1) * g;
  v = r.b2 * v + (1.f - r.b2) * g * g;
  const float denom = sqrtf(v / r.bc2) + r.eps;
  return p * (1.f - r.lr * r.wd) - r.lr * (m / r.bc1) / denom;
}

template <typename T>
__global__ __launch_bounds__(256) void adamw_kernel(AdamTensors a, AdamRates r, int count) {
  int t = 0;
  while (t + 1 < count && (int)blockIdx.x >= a.first[t + 1]) t++;
  const long n = a.n[t], i0 = (long)((int)blockIdx.x - a.first[t]) * PER_BLOCK;
  T* p = (T*)a.p[t];
  const T* g = (const T*)a.g[t];
  float *m = a.m[t], *v = a.v[t];
  if (a.vec >> t & 1) {
#pragma unroll
    for (int k = 0; k < PER_BLOCK; k += 256 * 8) {
      const long i = i0 + k + threadIdx.x * 8L;
      if (i + 8 <= n) {
        float pv[8], gv[8], mv[8], vv[8];
        ldv<8>(p + i, pv);
        ldv<8>(g + i, gv);
        ldv<8>(m + i, mv);
        ldv<8>(v + i, vv);
#pragma unroll
        for (int j = 0; j < 8; j++) pv[j] = adam_one(pv[j], gv[j], mv[j], vv[j], r);
        stv<8>(p + i, pv);
        stv<8>(m + i, mv);
        stv<8>(v + i, vv);
      } else {
        for (long e = i; e < n; e++) stf(p + e, adam_one(ldf(p + e), ldf(g + e), m[e], v[e], r));
      }
    }
    return;
  }
  for (long i = i0 + threadIdx.x; i < min(i0 + PER_BLOCK, n); i += 256)
    stf(p + i, adam_one(ldf(p + i), ldf(g + i), m[i], v[i], r));
}

// tensors of one dtype, all at the same step
void adamw_step_many(std::vector<torch::Tensor> p, std::vector<torch::Tensor> g,
                     std::vector<torch::Tensor> m, std::vector<torch::Tensor> v, double lr,
                     double b1, double b2, double eps, double wd, long step) {
  TORCH_CHECK(g.size() == p.size() && m.size() == p.size() && v.size() == p.size());
  if (p.empty()) return;
  const auto type = p[0].scalar_type();
  TORCH_CHECK(type == torch::kBFloat16 || type == torch::kFloat32);
  const AdamRates r{(float)lr, (float)b1, (float)b2, (float)eps, (float)wd,
                    1.f - powf((float)b1, (float)step), 1.f - powf((float)b2, (float)step)};
  auto stream = at::hip::getCurrentHIPStream();
  for (auto& t : g) t = t.contiguous();
  AdamTensors a;
  int count = 0;
  long blocks = 0;
  auto launch = [&] {
    if (count == 0) return;
    a.first[count] = (int)blocks;
    if (type == torch::kBFloat16)
      hipLaunchKernelGGL(adamw_kernel<short>, dim3(blocks), dim3(256), 0, stream, a, r, count);
    else
      hipLaunchKernelGGL(adamw_kernel<float>, dim3(blocks), dim3(256), 0, stream, a, r, count);
    HIP_CHECK_LAST();
    count = 0;
    blocks = 0;
  };
  for (size_t i = 0; i < p.size(); i++) {
    TORCH_CHECK(p[i].is_cuda() && g[i].is_cuda() && m[i].is_cuda() && v[i].is_cuda());
    TORCH_CHECK(p[i].is_contiguous() && m[i].is_contiguous() && v[i].is_contiguous());
    TORCH_CHECK(m[i].scalar_type() == torch::kFloat32 && v[i].scalar_type() == torch::kFloat32);
    TORCH_CHECK(p[i].scalar_type() == type && g[i].scalar_type() == type);
    const long n = p[i].numel();
    TORCH_CHECK(g[i].numel() == n && m[i].numel() == n && v[i].numel() == n);
    if (n == 0) continue;
    const long here = (n + PER_BLOCK - 1) / PER_BLOCK;
    TORCH_CHECK(here < (1L << 30), "tensor too large");
    if (count == AT_ONCE || blocks + here >= (1L << 30)) launch();
    if (count == 0) a.vec = 0;
    a.p[count] = p[i].data_ptr();
    a.g[count] = g[i].data_ptr();
    a.m[count] = m[i].data_ptr<float>();
    a.v[count] = v[i].data_ptr<float>();
    a.n[count] = n;
    a.first[count] = (int)blocks;
    if (((uintptr_t)a.p[count] | (uintptr_t)a.g[count] | (uintptr_t)a.m[count] |
         (uintptr_t)a.v[count]) % 16 == 0)
      a.vec |= 1ull << count;
    blocks += here;
    count++;
  }
  launch();
}

void adamw_step(torch::Tensor p, torch::Tensor g, torch::Tensor m, torch::Tensor v,
                double lr, double b1, double b2, double eps, double wd, long step) {
  adamw_step_many({p}, {g}, {m}, {v}, lr, b1, b2, eps, wd, step);
}
