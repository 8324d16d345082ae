// RMSNorm fwd/bwd, RoPE apply, SwiGLU fwd/bwd — fused memory-bound kernels
// for gfx950.  All bf16 I/O with fp32 accumulation, bf16x8 (16 B) vector
// loads per lane; the norms reduce a row in one workgroup or wave.
#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>

#include "common.h"
#include "checks.h"
#include "qkv.h"

// ------------------------------------------------------------- RMSNorm fwd
// x [N, H] bf16 -> y [N, H] bf16, invrms [N] f32.  One 256-thread block/row.
template <int BLOCK>
__global__ void rmsnorm_fwd_kernel(const short* __restrict__ x,
                                   const short* __restrict__ w,
                                   short* __restrict__ y,
                                   float* __restrict__ invrms,
                                   int H, float eps) {
  __shared__ float scratch[BLOCK / 64];
  const long row = blockIdx.x;
  const short* xr = x + row * (long)H;
  short* yr = y + row * (long)H;
  float ss = 0.f;
  const int nvec = H / 8;
  for (int i = threadIdx.x; i < nvec; i += BLOCK) {
    s16x8 v = *reinterpret_cast<const s16x8*>(xr + i * 8);
#pragma unroll
    for (int j = 0; j < 8; j++) { float f = bf2f(v[j]); ss += f * f; }
  }
  ss = block_sum<BLOCK>(ss, scratch);
  const float inv = rsqrtf(ss / (float)H + eps);
  if (threadIdx.x == 0) invrms[row] = inv;
  for (int i = threadIdx.x; i < nvec; i += BLOCK) {
    s16x8 v = *reinterpret_cast<const s16x8*>(xr + i * 8);
    s16x8 wv = *reinterpret_cast<const s16x8*>(w + i * 8);
    s16x8 o;
#pragma unroll
    for (int j = 0; j < 8; j++) {
      // match the reference numerics: bf16(x*inv) * w
      float t = bf2f(f2bf(bf2f(v[j]) * inv));
      o[j] = f2bf(t * bf2f(wv[j]));
    }
    *reinterpret_cast<s16x8*>(yr + i * 8) = o;
  }
}

// The first norm of a forward together with the lookup of its rows: h = table[ids], y = its norm,
// by rmsnorm_fwd_kernel's steps in its order; and, of a decode step, the place of each row's
// newest position (decode_inputs).  Bound by its launch and two dependent latencies where rows are
// few (three launches of 4.6 us in a decode step before: 12 rows, 2 layers and 82 tokens 16.9 ms,
// now 16.0), by memory where they are many.
struct Place {
  const int* lens;       // [N], or null
  const int* bt;         // [N, P]
  long* pos;
  long* slots;
  int P, ps;
};
template <int SL>        // vectors of 8 a thread
__global__ __launch_bounds__(256)
void embed_rms_norm_kernel(const long* __restrict__ ids, const short* __restrict__ table,
                           const short* __restrict__ w, short* __restrict__ h,
                           short* __restrict__ y, long V, int H, float eps, Place place) {
  __shared__ float scratch[4];
  const long row = blockIdx.x, id = ids[row];
  CUDA_KERNEL_ASSERT(id >= 0 && id < V);
  const short* xr = table + id * H;
  s16x8 v[SL];
  float ss = 0.f;
#pragma unroll
  for (int s = 0; s < SL; s++) {
    const int i = threadIdx.x + 256 * s;
    if (i < H / 8) v[s] = *reinterpret_cast<const s16x8*>(xr + i * 8);
  }
  if (place.lens && threadIdx.x == 0) {
    const int at = place.lens[row] - 1;
    place.pos[row] = at;
    place.slots[row] = (long)place.bt[row * place.P + min(max(at, 0) / place.ps, place.P - 1)] *
                           place.ps + max(at, 0) % place.ps;
  }
#pragma unroll
  for (int s = 0; s < SL; s++) {
    const int i = threadIdx.x + 256 * s;
    if (i >= H / 8) continue;
    *reinterpret_cast<s16x8*>(h + row * H + i * 8) = v[s];
#pragma unroll
    for (int j = 0; j < 8; j++) { float f = bf2f(v[s][j]); ss += f * f; }
  }
  ss = block_sum<256>(ss, scratch);
  const float inv = rsqrtf(ss / (float)H + eps);
#pragma unroll
  for (int s = 0; s < SL; s++) {
    const int i = threadIdx.x + 256 * s;
    if (i >= H / 8) continue;
    const s16x8 wv = *reinterpret_cast<const s16x8*>(w + i * 8);
    s16x8 o;
#pragma unroll
    for (int j = 0; j < 8; j++) o[j] = f2bf(bf2f(f2bf(bf2f(v[s][j]) * inv)) * bf2f(wv[j]));
    *reinterpret_cast<s16x8*>(y + row * H + i * 8) = o;
  }
}

// ------------------------------------------------------------- RMSNorm bwd
// dx = inv * (g - x_hat * mean(g * x_hat)) [+ extra],  g = dy*w,  x_hat = x*inv
// `extra` is what the residual stream's later consumers add to dx.  A row is held
// in registers between the mean and dx: by one wave up to H = 2048 (no barrier),
// else by the workgroup.  With DW, a workgroup sums dw over its rows and leaves
// the sums in part [workgroups, H] for rmsnorm_dw_kernel: no atomics, one order.
//
// Bound by memory: three or four passes over [N, H].  48720 x 1536 without dw: 96 us
// with the addition, where reading every row twice and 1024 workgroups'
// atomics on dw took 306 and the addition 75 more.
template <int WAVES, int SL, bool DW>     // waves of a row, vectors of 8 per lane
__global__ __launch_bounds__(256)
void rmsnorm_bwd_kernel(const short* __restrict__ dy,
                        const short* __restrict__ x,
                        const short* __restrict__ w,
                        const float* __restrict__ invrms,
                        const short* __restrict__ extra,   // or null
                        short* __restrict__ dx,
                        float* __restrict__ part,
                        long N, int H) {
  __shared__ float scratch[4];
  __shared__ float sums[DW && WAVES == 1 ? 4 * 64 * SL * 8 : 1];
  constexpr int LANES = 64 * WAVES, ROWS = 4 / WAVES;
  const int nvec = H / 8, l = threadIdx.x % LANES;
  float dwacc[SL][8];
  s16x8 wv[SL];
#pragma unroll
  for (int k = 0; k < SL; k++) {
    const int i = l + LANES * k;
    wv[k] = i < nvec ? *reinterpret_cast<const s16x8*>(w + i * 8) : s16x8{};
#pragma unroll
    for (int j = 0; j < 8; j++) dwacc[k][j] = 0.f;
  }
  for (long row = (long)blockIdx.x * ROWS + threadIdx.x / LANES;
       WAVES > 1 ? row < N : row - threadIdx.x / LANES < N; row += (long)gridDim.x * ROWS) {
    const bool ok = row < N;
    const long at = min(row, N - 1) * H;
    const float inv = invrms[min(row, N - 1)];
    s16x8 dv[SL], xv[SL], ev[SL];
    float dot = 0.f;
#pragma unroll
    for (int k = 0; k < SL; k++) {
      const int i = l + LANES * k;
      if (i < nvec) {
        dv[k] = *reinterpret_cast<const s16x8*>(dy + at + i * 8);
        xv[k] = *reinterpret_cast<const s16x8*>(x + at + i * 8);
        if (extra) ev[k] = *reinterpret_cast<const s16x8*>(extra + at + i * 8);
      }
    }
#pragma unroll
    for (int k = 0; k < SL; k++)
      if (l + LANES * k < nvec)
#pragma unroll
        for (int j = 0; j < 8; j++) dot += bf2f(dv[k][j]) * bf2f(wv[k][j]) * bf2f(xv[k][j]) * inv;
    dot = (WAVES == 1 ? wave_sum(dot) : block_sum<256>(dot, scratch)) / (float)H;
    if (!ok) continue;
#pragma unroll
    for (int k = 0; k < SL; k++) {
      const int i = l + LANES * k;
      if (i >= nvec) continue;
      s16x8 o;
#pragma unroll
      for (int j = 0; j < 8; j++) {
        const float xh = bf2f(xv[k][j]) * inv;
        const float g = bf2f(dv[k][j]) * bf2f(wv[k][j]);
        const float d = (g - xh * dot) * inv;
        o[j] = f2bf(extra ? d + bf2f(ev[k][j]) : d);
        if (DW) dwacc[k][j] += bf2f(dv[k][j]) * bf2f(f2bf(xh));
      }
      *reinterpret_cast<s16x8*>(dx + at + i * 8) = o;
    }
  }
  if constexpr (DW) {
    float* out = part + (long)blockIdx.x * H;
    if constexpr (WAVES == 1) {
#pragma unroll
      for (int k = 0; k < SL; k++)
#pragma unroll
        for (int j = 0; j < 8; j++) sums[(threadIdx.x / 64 * SL + k) * 512 + j * 64 + l] = dwacc[k][j];
      __syncthreads();
      for (int i = threadIdx.x; i < H; i += 256) {
        const int v = i / 8, at = v / 64 * 512 + i % 8 * 64 + v % 64;
        float t = 0.f;
        for (int q = 0; q < 4; q++) t += sums[q * SL * 512 + at];
        out[i] = t;
      }
    } else {
#pragma unroll
      for (int k = 0; k < SL; k++)
        if (l + LANES * k < nvec) stv<8>(out + (l + LANES * k) * 8, dwacc[k]);
    }
  }
}

// column sums of part [n, H]: 64 columns per workgroup, 16 rows at a time
__global__ __launch_bounds__(1024) void rmsnorm_dw_kernel(const float* __restrict__ part,
                                                          short* __restrict__ dw, int n, int H) {
  __shared__ float sums[16][64];
  const int c = blockIdx.x * 64 + (threadIdx.x & 63), r = threadIdx.x >> 6;
  float t = 0.f;
  if (c < H)
    for (int i = r; i < n; i += 16) t += part[(long)i * H + c];
  sums[r][threadIdx.x & 63] = t;
  __syncthreads();
  if (r == 0 && c < H) {
    for (int i = 1; i < 16; i++) t += sums[i][threadIdx.x];
    dw[c] = f2bf(t);
  }
}

// ----------------------------------------------------------------- RoPE
// x [T, Hh, D] bf16 in-place; table [maxpos, D] f32 (cos | sin halves);
// positions [T] i64.  sign=-1 applies the inverse rotation (backward).
__global__ void rope_kernel(const short* __restrict__ x,
                            short* __restrict__ y,
                            const float* __restrict__ table,
                            const long* __restrict__ pos,
                            int T, int Hh, int D, float sign) {
  // one thread per (t, h, 4 pairs)
  const int pairs4 = D / 8;  // groups of 4 rotation pairs
  long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const long total = (long)T * Hh * pairs4;
  if (idx >= total) return;
  const int g = idx % pairs4;
  const int h = (idx / pairs4) % Hh;
  const long t = idx / ((long)pairs4 * Hh);
  const short* base = x + (t * Hh + h) * (long)D;
  short* obase = y + (t * Hh + h) * (long)D;
  const float* tb = table + pos[t] * (long)D;
  s16x4 x1 = *reinterpret_cast<const s16x4*>(base + g * 4);
  s16x4 x2 = *reinterpret_cast<const s16x4*>(base + D / 2 + g * 4);
  f32x4 c = *reinterpret_cast<const f32x4*>(tb + g * 4);
  f32x4 s = *reinterpret_cast<const f32x4*>(tb + D / 2 + g * 4);
  s16x4 o1, o2;
#pragma unroll
  for (int j = 0; j < 4; j++) {
    float a = bf2f(x1[j]), b = bf2f(x2[j]);
    float cs = c[j], sn = s[j] * sign;
    o1[j] = f2bf(a * cs - b * sn);
    o2[j] = f2bf(b * cs + a * sn);
  }
  *reinterpret_cast<s16x4*>(obase + g * 4) = o1;
  *reinterpret_cast<s16x4*>(obase + D / 2 + g * 4) = o2;
}

// ----------------------------------------------------------------- SwiGLU
// gate_up [N, 2I] -> y [N, I]; y = silu(g) * u
__global__ void swiglu_fwd_kernel(const short* __restrict__ gu,
                                  short* __restrict__ y,
                                  long N, int I) {
  long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;  // in units of 8
  const long total = N * (long)(I / 8);
  if (idx >= total) return;
  const long n = idx / (I / 8);
  const int i = (idx % (I / 8)) * 8;
  const short* row = gu + n * 2L * I;
  s16x8 g = *reinterpret_cast<const s16x8*>(row + i);
  s16x8 u = *reinterpret_cast<const s16x8*>(row + I + i);
  s16x8 o;
#pragma unroll
  for (int j = 0; j < 8; j++) {
    float gf = bf2f(g[j]);
    float sig = 1.f / (1.f + __expf(-gf));
    o[j] = f2bf(gf * sig * bf2f(u[j]));
  }
  *reinterpret_cast<s16x8*>(y + n * (long)I + i) = o;
}

__global__ void swiglu_bwd_kernel(const short* __restrict__ dy,
                                  const short* __restrict__ gu,
                                  short* __restrict__ dgu,
                                  long N, int I) {
  long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const long total = N * (long)(I / 8);
  if (idx >= total) return;
  const long n = idx / (I / 8);
  const int i = (idx % (I / 8)) * 8;
  const short* row = gu + n * 2L * I;
  s16x8 g = *reinterpret_cast<const s16x8*>(row + i);
  s16x8 u = *reinterpret_cast<const s16x8*>(row + I + i);
  s16x8 d = *reinterpret_cast<const s16x8*>(dy + n * (long)I + i);
  s16x8 dg, du;
#pragma unroll
  for (int j = 0; j < 8; j++) {
    float gf = bf2f(g[j]), uf = bf2f(u[j]), df = bf2f(d[j]);
    float sig = 1.f / (1.f + __expf(-gf));
    float silu = gf * sig;
    float dsilu = sig * (1.f + gf * (1.f - sig));
    dg[j] = f2bf(df * uf * dsilu);
    du[j] = f2bf(df * silu);
  }
  short* drow = dgu + n * 2L * I;
  *reinterpret_cast<s16x8*>(drow + i) = dg;
  *reinterpret_cast<s16x8*>(drow + I + i) = du;
}

// ======================================================== host wrappers ==
static inline void check_bf16(const torch::Tensor& t, const char* name) {
  TORCH_CHECK(t.is_cuda() && t.scalar_type() == torch::kBFloat16, name, " must be bf16 on GPU");
  TORCH_CHECK(t.is_contiguous(), name, " must be contiguous");
}

std::vector<torch::Tensor> rmsnorm_fwd(torch::Tensor x, torch::Tensor w, double eps) {
  check_bf16(x, "x"); check_bf16(w, "w");
  const int H = x.size(-1);
  TORCH_CHECK(H % 8 == 0, "hidden size must be divisible by 8");
  const long N = x.numel() / H;
  auto y = torch::empty_like(x);
  auto invrms = torch::empty({N}, x.options().dtype(torch::kFloat32));
  auto stream = at::hip::getCurrentHIPStream();
  hipLaunchKernelGGL((rmsnorm_fwd_kernel<256>), dim3(N), dim3(256), 0, stream,
                     (const short*)x.data_ptr(), (const short*)w.data_ptr(),
                     (short*)y.data_ptr(), invrms.data_ptr<float>(), H, (float)eps);
  HIP_CHECK_LAST();
  return {y, invrms};
}

// (y, h[, positions, slots]): the norm of h = table[ids], and with lens and bt decode_inputs'
// result.
std::vector<torch::Tensor> embed_rms_norm(torch::Tensor ids, torch::Tensor table, torch::Tensor w,
                                          double eps, c10::optional<torch::Tensor> lens,
                                          c10::optional<torch::Tensor> bt, long page_size) {
  on_gpu({ids, table, w, lens, bt});
  check_bf16(table, "table"); check_bf16(w, "w");
  TORCH_CHECK(ids.scalar_type() == torch::kLong && ids.is_contiguous() && ids.dim() == 1 &&
              table.dim() == 2, "embed_rms_norm: ids [T], table [V, H]");
  const long N = ids.size(0), V = table.size(0), H = table.size(1);
  TORCH_CHECK(H % 8 == 0 && H > 0 && H <= 8192 && w.numel() == H && N < (1L << 31),
              "embed_rms_norm: sizes");
  TORCH_CHECK((uintptr_t)table.data_ptr() % 16 == 0 && (uintptr_t)w.data_ptr() % 16 == 0,
              "embed_rms_norm: alignment");
  auto y = torch::empty({N, H}, table.options()), h = torch::empty_like(y);
  std::vector<torch::Tensor> out{y, h};
  Place place{};
  if (lens) {
    TORCH_CHECK(bt && bt->dim() == 2 && bt->size(0) == N && bt->size(1) > 0 && page_size > 0 &&
                lens->numel() == N && lens->scalar_type() == at::kInt && lens->is_contiguous() &&
                bt->scalar_type() == at::kInt && bt->is_contiguous(),
                "embed_rms_norm: contiguous int32 lengths [T], pages [T, P]");
    for (int i = 0; i < 2; i++) out.push_back(torch::empty({N}, ids.options()));
    place = {lens->data_ptr<int>(), bt->data_ptr<int>(), out[2].data_ptr<long>(),
             out[3].data_ptr<long>(), (int)bt->size(1), (int)page_size};
  }
  if (N == 0) return out;
#define LAUNCH(SL)                                                                             \
  hipLaunchKernelGGL((embed_rms_norm_kernel<SL>), dim3(N), dim3(256), 0,                       \
                     at::hip::getCurrentHIPStream(), ids.data_ptr<long>(),                     \
                     (const short*)table.data_ptr(), (const short*)w.data_ptr(),               \
                     (short*)h.data_ptr(), (short*)y.data_ptr(), V, (int)H, (float)eps, place)
  if (H <= 2048) LAUNCH(1);
  else if (H <= 4096) LAUNCH(2);
  else LAUNCH(4);
#undef LAUNCH
  HIP_CHECK_LAST();
  return out;
}

// dx and, if wanted, dw (else an empty tensor).  extra: added to dx.
std::vector<torch::Tensor> rmsnorm_bwd(torch::Tensor dy, torch::Tensor x,
                                       torch::Tensor w, torch::Tensor invrms,
                                       c10::optional<torch::Tensor> extra, bool want_dw) {
  check_bf16(dy, "dy"); check_bf16(x, "x"); check_bf16(w, "w");
  const int H = x.size(-1);
  const long N = x.numel() / H;
  TORCH_CHECK(H % 8 == 0 && H <= 256 * 8 * 4, "hidden too large for rmsnorm_bwd slices");
  TORCH_CHECK(dy.sizes() == x.sizes() && w.numel() == H && invrms.numel() == N);
  const short* ep = nullptr;
  if (extra.has_value()) {
    check_bf16(*extra, "extra");
    TORCH_CHECK(extra->sizes() == x.sizes());
    ep = (const short*)extra->data_ptr();
  }
  auto dx = torch::empty_like(x);
  auto dw = want_dw ? torch::empty({H}, x.options()) : torch::empty({0}, x.options());
  if (N == 0) return {dx, want_dw ? dw.zero_() : dw};
  auto stream = at::hip::getCurrentHIPStream();
  // without dw a workgroup per row (or four); with it, 512 share the rows
  const long most = (N + (H <= 2048 ? 3 : 0)) / (H <= 2048 ? 4 : 1);
  const long grid = want_dw ? std::min<long>(most, 512) : std::min<long>(most, 1 << 20);
  torch::Tensor part;
  if (want_dw) part = torch::empty({grid, H}, x.options().dtype(torch::kFloat32));
  float* pp = want_dw ? part.data_ptr<float>() : nullptr;
#define LAUNCH(WAVES, SL, DW)                                                             \
  hipLaunchKernelGGL((rmsnorm_bwd_kernel<WAVES, SL, DW>), dim3(grid), dim3(256), 0, stream, \
                     (const short*)dy.data_ptr(), (const short*)x.data_ptr(),             \
                     (const short*)w.data_ptr(), invrms.data_ptr<float>(), ep,            \
                     (short*)dx.data_ptr(), pp, N, H)
#define LAUNCH_DW(WAVES, SL) do { if (want_dw) LAUNCH(WAVES, SL, true); else LAUNCH(WAVES, SL, false); } while (0)
  if (H <= 512) LAUNCH_DW(1, 1);
  else if (H <= 1024) LAUNCH_DW(1, 2);
  else if (H <= 2048) LAUNCH_DW(1, 4);
  else if (H <= 4096) LAUNCH_DW(4, 2);
  else LAUNCH_DW(4, 4);
#undef LAUNCH_DW
#undef LAUNCH
  if (want_dw)
    hipLaunchKernelGGL(rmsnorm_dw_kernel, dim3((H + 63) / 64), dim3(1024), 0, stream, pp,
                       (short*)dw.data_ptr(), (int)grid, H);
  HIP_CHECK_LAST();
  return {dx, dw};
}

torch::Tensor rope_fwd(torch::Tensor x, torch::Tensor table, torch::Tensor positions,
                       double sign) {
  check_bf16(x, "x");
  on_gpu({table, positions});
  TORCH_CHECK(table.scalar_type() == torch::kFloat32, "rope table must be fp32");
  TORCH_CHECK(positions.scalar_type() == torch::kLong, "positions must be int64");
  const int D = x.size(-1);
  const int Hh = x.size(1);
  const int T = x.size(0);
  TORCH_CHECK(D % 8 == 0, "head_dim must be divisible by 8");
  const long total = (long)T * Hh * (D / 8);
  const int block = 256;
  const long grid = (total + block - 1) / block;
  auto y = torch::empty_like(x);
  auto stream = at::hip::getCurrentHIPStream();
  hipLaunchKernelGGL(rope_kernel, dim3(grid), dim3(block), 0, stream,
                     (const short*)x.data_ptr(), (short*)y.data_ptr(),
                     table.data_ptr<float>(),
                     positions.data_ptr<long>(), T, Hh, D, (float)sign);
  HIP_CHECK_LAST();
  return y;
}

static void check_rope(const torch::Tensor& table, const torch::Tensor& positions, long T, int D) {
  on_gpu({table, positions});
  TORCH_CHECK(table.scalar_type() == torch::kFloat32 && table.is_contiguous() &&
              table.size(-1) == D, "rope table must be fp32 [positions, head_dim]");
  TORCH_CHECK(positions.scalar_type() == torch::kLong && positions.is_contiguous() &&
              positions.numel() == T, "positions must be int64, one per token");
  TORCH_CHECK(D % 16 == 0, "head_dim must be divisible by 16");
}

// qkv [T, (Hq + 2 Hkv) D] -> q [T, Hq, D], k and v [T, Hkv, D], q and k rotated
std::vector<torch::Tensor> qkv_rope_fwd(torch::Tensor qkv, torch::Tensor table,
                                        torch::Tensor positions, long Hq, long Hkv) {
  check_bf16(qkv, "qkv");
  TORCH_CHECK(qkv.dim() == 2 && Hq > 0 && Hkv > 0 && qkv.size(1) % (Hq + 2 * Hkv) == 0);
  const long T = qkv.size(0), D = qkv.size(1) / (Hq + 2 * Hkv);
  check_rope(table, positions, T, (int)D);
  if ((uintptr_t)qkv.data_ptr() % 16) qkv = qkv.clone();
  auto q = torch::empty({T, Hq, D}, qkv.options());
  auto k = torch::empty({T, Hkv, D}, qkv.options()), v = torch::empty_like(k);
  auto stream = at::hip::getCurrentHIPStream();
  by_tokens(T, (Hq + 2 * Hkv) * (D / 16), [&](long t0, unsigned units) {
    QkvRope a{};
    a.qkv = (const short*)qkv.data_ptr() + t0 * qkv.size(1);
    a.q = (short*)q.data_ptr() + t0 * Hq * D;
    a.k = (short*)k.data_ptr() + t0 * Hkv * D;
    a.v = (short*)v.data_ptr() + t0 * Hkv * D;
    a.table = table.data_ptr<float>();
    a.pos = positions.data_ptr<long>() + t0;
    a.Hq = Hq;
    a.Hkv = Hkv;
    a.D = D;
    hipLaunchKernelGGL(qkv_rope_kernel<void>, dim3((units + 255) / 256), dim3(256), 0, stream, a,
                       units);
  });
  HIP_CHECK_LAST();
  return {q, k, v};
}

torch::Tensor qkv_rope_bwd(c10::optional<torch::Tensor> dq, c10::optional<torch::Tensor> dk,
                           c10::optional<torch::Tensor> dv, torch::Tensor table,
                           torch::Tensor positions, long Hq, long Hkv) {
  const long T = positions.numel(), D = table.size(-1);
  check_rope(table, positions, T, (int)D);
  auto ptr = [&](c10::optional<torch::Tensor>& x, long H) -> const short* {
    if (!x.has_value()) return nullptr;
    check_bf16(*x, "gradient");
    TORCH_CHECK(x->numel() == T * H * D, "gradient has another shape");
    if ((uintptr_t)x->data_ptr() % 16) x = x->clone();
    return (const short*)x->data_ptr();
  };
  const short *q = ptr(dq, Hq), *k = ptr(dk, Hkv), *v = ptr(dv, Hkv);
  auto out = torch::empty({T, (Hq + 2 * Hkv) * D}, table.options().dtype(torch::kBFloat16));
  auto stream = at::hip::getCurrentHIPStream();
  by_tokens(T, (Hq + 2 * Hkv) * (D / 16), [&](long t0, unsigned units) {
    auto from = [&](const short* p, long H) { return p ? p + t0 * H * D : nullptr; };
    hipLaunchKernelGGL(qkv_rope_bwd_kernel, dim3((units + 255) / 256), dim3(256), 0, stream,
                       from(q, Hq), from(k, Hkv), from(v, Hkv), table.data_ptr<float>(),
                       positions.data_ptr<long>() + t0,
                       (short*)out.data_ptr() + t0 * (Hq + 2 * Hkv) * D, (int)Hq, (int)Hkv, (int)D,
                       units);
  });
  HIP_CHECK_LAST();
  return out;
}

torch::Tensor swiglu_fwd(torch::Tensor gu) {
  check_bf16(gu, "gate_up");
  const int I2 = gu.size(-1);
  TORCH_CHECK(I2 % 16 == 0, "2*intermediate must be divisible by 16");
  const int I = I2 / 2;
  const long N = gu.numel() / I2;
  auto y = torch::empty({gu.size(0), I}, gu.options());
  const long total = N * (I / 8);
  const int block = 256;
  auto stream = at::hip::getCurrentHIPStream();
  hipLaunchKernelGGL(swiglu_fwd_kernel, dim3((total + block - 1) / block), dim3(block),
                     0, stream, (const short*)gu.data_ptr(), (short*)y.data_ptr(), N, I);
  HIP_CHECK_LAST();
  return y;
}

torch::Tensor swiglu_bwd(torch::Tensor dy, torch::Tensor gu) {
  check_bf16(dy, "dy"); check_bf16(gu, "gate_up");
  const int I2 = gu.size(-1);
  const int I = I2 / 2;
  const long N = gu.numel() / I2;
  auto dgu = torch::empty_like(gu);
  const long total = N * (I / 8);
  const int block = 256;
  auto stream = at::hip::getCurrentHIPStream();
  hipLaunchKernelGGL(swiglu_bwd_kernel, dim3((total + block - 1) / block), dim3(block),
                     0, stream, (const short*)dy.data_ptr(), (const short*)gu.data_ptr(),
                     (short*)dgu.data_ptr(), N, I);
  HIP_CHECK_LAST();
  return dgu;
}

// ----------------------------------------------- fused residual + RMSNorm
// h = x + res;  y = rmsnorm(h) * w.  For H <= BLOCK*8 each thread keeps its
// h slice in registers across both phases (read x,res; write h,y — the
// unfused pair costs an extra h read plus a launch).  invrms saved for the
// backward, which reuses rmsnorm_bwd on h (d h = d x = d res).
//
// Where few rows decode it is a chain of latencies: the weight is asked for with the rows
// and the sum crosses the waves with one barrier.  With `splits` x is 32-bit parts of the
// depth of the product before ([splits][rows][H]) that are added up here, for which that
// product took another launch: 64 rows of 1536 in 5 parts 4.5 us, where the sum took 4.6
// and this 4.7.
template <int BLOCK>
DEVINL float block_sum_once(float v, float* scratch) {
  static_assert(BLOCK == 256, "four waves");
  v = wave_sum(v);
  if ((threadIdx.x & 63) == 0) scratch[threadIdx.x >> 6] = v;
  __syncthreads();
  return (scratch[0] + scratch[2]) + (scratch[1] + scratch[3]);
}
template <int BLOCK, bool PARTS>
__global__ void rmsnorm_addres_fwd_kernel(const void* __restrict__ x,
                                          const short* __restrict__ res,
                                          const short* __restrict__ w,
                                          short* __restrict__ h,
                                          short* __restrict__ y,
                                          float* __restrict__ invrms,
                                          int H, float eps, int splits) {
  __shared__ float scratch[BLOCK / 64];
  const long row = blockIdx.x, part = (long)gridDim.x * H;
  auto load_x = [&](int i) {
    if constexpr (PARTS)
      return sum_parts8((const float*)x + row * (long)H + i * 8, part, splits, nullptr);
    else
      return *reinterpret_cast<const s16x8*>((const short*)x + row * (long)H + i * 8);
  };
  const short* rr = res + row * (long)H;
  short* hr = h + row * (long)H;
  short* yr = y + row * (long)H;
  const int nvec = H / 8;
  float ss = 0.f;
  if (nvec <= BLOCK) {
    // register-resident path (H <= BLOCK*8)
    s16x8 hv{}, wv{};
    const int i = threadIdx.x;
    if (i < nvec) {
      s16x8 rv = *reinterpret_cast<const s16x8*>(rr + i * 8);
      wv = *reinterpret_cast<const s16x8*>(w + i * 8);
      s16x8 xv = load_x(i);
#pragma unroll
      for (int j = 0; j < 8; j++) {
        const float f = bf2f(xv[j]) + bf2f(rv[j]);
        hv[j] = f2bf(f);
        const float fb = bf2f(hv[j]);
        ss += fb * fb;
      }
    }
    ss = block_sum_once<BLOCK>(ss, scratch);
    const float inv = rsqrtf(ss / (float)H + eps);
    if (invrms && threadIdx.x == 0) invrms[row] = inv;
    if (i < nvec) {
      s16x8 o;
#pragma unroll
      for (int j = 0; j < 8; j++) {
        const float t = bf2f(f2bf(bf2f(hv[j]) * inv));
        o[j] = f2bf(t * bf2f(wv[j]));
      }
      *reinterpret_cast<s16x8*>(hr + i * 8) = hv;
      *reinterpret_cast<s16x8*>(yr + i * 8) = o;
    }
    return;
  }
  // general path: write h in pass 1, re-read (L2-hot) in pass 2
  for (int i = threadIdx.x; i < nvec; i += BLOCK) {
    s16x8 rv = *reinterpret_cast<const s16x8*>(rr + i * 8);
    s16x8 xv = load_x(i);
    s16x8 hv;
#pragma unroll
    for (int j = 0; j < 8; j++) {
      hv[j] = f2bf(bf2f(xv[j]) + bf2f(rv[j]));
      const float f = bf2f(hv[j]);
      ss += f * f;
    }
    *reinterpret_cast<s16x8*>(hr + i * 8) = hv;
  }
  ss = block_sum<BLOCK>(ss, scratch);
  const float inv = rsqrtf(ss / (float)H + eps);
  if (invrms && threadIdx.x == 0) invrms[row] = inv;
  for (int i = threadIdx.x; i < nvec; i += BLOCK) {
    s16x8 hv = *reinterpret_cast<const s16x8*>(hr + i * 8);
    s16x8 wv = *reinterpret_cast<const s16x8*>(w + i * 8);
    s16x8 o;
#pragma unroll
    for (int j = 0; j < 8; j++) {
      const float t = bf2f(f2bf(bf2f(hv[j]) * inv));
      o[j] = f2bf(t * bf2f(wv[j]));
    }
    *reinterpret_cast<s16x8*>(yr + i * 8) = o;
  }
}

std::vector<torch::Tensor> rmsnorm_addres_fwd(torch::Tensor x, torch::Tensor res,
                                              torch::Tensor w, double eps) {
  on_gpu({x, res, w});
  TORCH_CHECK(x.scalar_type() == torch::kBFloat16);
  TORCH_CHECK(x.is_contiguous() && res.is_contiguous() && w.is_contiguous());
  TORCH_CHECK(x.sizes() == res.sizes());
  const long N = x.numel() / x.size(-1);
  const int H = x.size(-1);
  TORCH_CHECK(H % 8 == 0);
  auto h = torch::empty_like(x);
  auto y = torch::empty_like(x);
  auto invrms = torch::empty({N}, x.options().dtype(torch::kFloat32));
  if (N == 0) return {y, h, invrms};
  auto stream = at::hip::getCurrentHIPStream();
  hipLaunchKernelGGL((rmsnorm_addres_fwd_kernel<256, false>), dim3(N), dim3(256), 0, stream,
                     x.data_ptr(), (const short*)res.data_ptr(),
                     (const short*)w.data_ptr(), (short*)h.data_ptr(),
                     (short*)y.data_ptr(), invrms.data_ptr<float>(), H, (float)eps, 0);
  HIP_CHECK_LAST();
  return {y, h, invrms};
}

// parts [splits, N, H] float32, res [N, H]: (rmsnorm(h) * w, h), h = sum of the parts + res
std::vector<torch::Tensor> rmsnorm_parts_fwd(torch::Tensor parts, torch::Tensor res,
                                             torch::Tensor w, double eps) {
  on_gpu({parts, res, w});
  TORCH_CHECK(parts.dim() == 3 && parts.scalar_type() == torch::kFloat32 &&
              parts.is_contiguous() && parts.size(0) > 0 && parts.size(0) <= 8,
              "rmsnorm_parts: float32 parts [1 to 8, rows, width]");
  const long N = parts.size(1), H = parts.size(2);
  TORCH_CHECK(res.scalar_type() == torch::kBFloat16 && res.is_contiguous() && res.dim() == 2 &&
              res.size(0) == N && res.size(1) == H && w.scalar_type() == torch::kBFloat16 &&
              w.is_contiguous() && w.numel() == H && H % 8 == 0, "rmsnorm_parts: bf16 [N, H]");
  for (const auto& t : {parts, res, w})
    TORCH_CHECK((uintptr_t)t.data_ptr() % 16 == 0, "rmsnorm_parts: operands on 16 bytes");
  auto h = torch::empty_like(res), y = torch::empty_like(res);
  if (N == 0) return {y, h};
  hipLaunchKernelGGL((rmsnorm_addres_fwd_kernel<256, true>), dim3(N), dim3(256), 0,
                     at::hip::getCurrentHIPStream(), parts.data_ptr(),
                     (const short*)res.data_ptr(), (const short*)w.data_ptr(),
                     (short*)h.data_ptr(), (short*)y.data_ptr(), nullptr, (int)H, (float)eps,
                     (int)parts.size(0));
  HIP_CHECK_LAST();
  return {y, h};
}

// ------------------------------------------------------ embedding's gradient
// out [V, H] += the rows of dy [T, H] that ids [T] name, 32-bit sums in a fixed order.  A
// workgroup a token: it marks the tokens of the same id in LDS, leaves if one of them comes
// before its own, and else lists and adds up all of them, as many side by side as its threads
// have columns for; nothing is sorted and nobody adds to the same row.  torch / this in us,
// with the zeros, over random ids: 212 x 896 17 / 8, 2667 x 896 143 / 18, 4096 x 1536 96 / 34;
// with a third of the tokens of one id 2667 x 896 145 / 34, 4096 x 1536 113 / 98.
constexpr int EMBED_MOST = 8192;       // tokens: a bit each in LDS, and T reads of ids by T
constexpr int EMBED_BLOCK = 512;

__global__ __launch_bounds__(EMBED_BLOCK)
void embedding_grad_kernel(const long* __restrict__ ids, const short* __restrict__ dy,
                           short* __restrict__ out, int T, int V, int H) {
  __shared__ unsigned long long same[EMBED_MOST / 64];
  __shared__ unsigned short list[EMBED_MOST];
  __shared__ int count;
  __shared__ __attribute__((aligned(16))) float sums[EMBED_BLOCK][8];
  const int t = blockIdx.x, tid = threadIdx.x, lane = tid & 63;
  const long id = ids[t];
  if (id < 0 || id >= V) return;
  bool before = false;
  for (int s0 = tid & ~63; s0 < T; s0 += EMBED_BLOCK) {
    const int s = s0 + lane;
    const unsigned long long m = __ballot(s < T && ids[s] == id);
    if (lane == 0) same[s0 / 64] = m;
    before |= s0 <= t && (m & (t - s0 >= 64 ? ~0ull : (1ull << (t - s0)) - 1)) != 0;
  }
  if (__syncthreads_or(before)) return;
  if (tid < 64) {                      // two words a lane
    unsigned long long m[2];
    int n = 0;
#pragma unroll
    for (int k = 0; k < 2; k++) {
      m[k] = (2 * lane + k) * 64 < T ? same[2 * lane + k] : 0;
      n += __popcll(m[k]);
    }
    int at = n;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int x = __shfl_up(at, off);
      if (lane >= off) at += x;
    }
    if (lane == 63) count = at;
    at -= n;
#pragma unroll
    for (int k = 0; k < 2; k++)
      for (; m[k]; m[k] &= m[k] - 1) list[at++] = 64 * (2 * lane + k) + __ffsll(m[k]) - 1;
  }
  __syncthreads();
  const int n = count, wide = H / 8, groups = max(1, EMBED_BLOCK / wide);
  const int g = tid / wide;            // every groups-th of the list
  for (int c = tid % wide; c < wide && g < groups; c += EMBED_BLOCK) {
    float sum[8] = {};
    constexpr int U = 8;
    for (int i = g; i < n; i += groups * U) {
      s16x8 v[U];
#pragma unroll
      for (int k = 0; k < U; k++)
        v[k] = *reinterpret_cast<const s16x8*>(
            dy + (long)list[min(i + groups * k, n - 1)] * H + 8 * c);
#pragma unroll
      for (int k = 0; k < U; k++) {
        if (i + groups * k >= n) continue;
#pragma unroll
        for (int j = 0; j < 8; j++) sum[j] += bf2f(v[k][j]);
      }
    }
    if (groups == 1 || n == 1) {
      if (g == 0) stv<8>(out + id * H + 8 * c, sum);
    } else {
      stv<8>(sums[tid], sum);
    }
  }
  if (groups == 1 || n == 1) return;
  __syncthreads();
  if (tid >= wide) return;
  float sum[8] = {};
  for (int k = 0; k < min(groups, n); k++) {
#pragma unroll
    for (int j = 0; j < 8; j++) sum[j] += sums[k * wide + tid][j];
  }
  stv<8>(out + id * H + 8 * tid, sum);
}

// the gradient of a [V, H] embedding whose rows ids [T] were looked up
torch::Tensor embedding_grad(torch::Tensor ids, torch::Tensor dy, long V) {
  on_gpu({ids, dy});
  TORCH_CHECK(ids.dim() == 1 && ids.scalar_type() == torch::kLong && ids.is_contiguous() &&
              dy.dim() == 2 && dy.scalar_type() == torch::kBFloat16 && dy.is_contiguous() &&
              dy.size(0) == ids.size(0) && (uintptr_t)dy.data_ptr() % 16 == 0,
              "embedding_grad: int64 ids [T], bf16 gradients [T, H]");
  const long T = ids.size(0), H = dy.size(1);
  TORCH_CHECK(T <= EMBED_MOST && H % 8 == 0 && H < (1L << 30) && V > 0 && V < (1L << 31),
              "embedding_grad: at most ", EMBED_MOST, " tokens, a width of 8");
  auto out = torch::zeros({V, H}, dy.options());
  if (T && H)
    hipLaunchKernelGGL(embedding_grad_kernel, dim3(T), dim3(EMBED_BLOCK), 0,
                       at::hip::getCurrentHIPStream(), ids.data_ptr<long>(),
                       (const short*)dy.data_ptr(), (short*)out.data_ptr(), (int)T, (int)V, (int)H);
  HIP_CHECK_LAST();
  return out;
}
