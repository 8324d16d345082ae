// Gradients of a rank-64 adapter: dA = du^T x [64, K] and dB = dy^T u [N, 64], both
// sums over all tokens, in one launch (and one that adds the parts).
//
// Bound by reading x and dy once.  A workgroup owns 128 of their columns and a part
// of the tokens, 64 at a time, which two LDS buffers receive by direct loads; both
// operands of the product are read transposed.  Few columns are divided among many
// parts, whose 32-bit sums lora_grad_sum_kernel adds in order.  48720 tokens, dB of N =
// 1536 54 us (floor 31), the library 150; of 17920 352 against 354; 8000 tokens of 1536 16
// against 54; 240 7 against 8, and 7.6 against 45 with the host's part of both products.
#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>

#include "common.h"
#include "checks.h"
#include "lds_tiles.h"

constexpr int RANK = 64, COLS = 128;

struct GradJob {
  const short *z, *v;      // [M, C] and [M, 64]; the result is z^T v or its transpose
  short* out;              // [C, 64], or [64, C] if `flat`
  float* part;             // [splits] of the same, if splits > 1
  int C, tiles, splits, flat;
};

__global__ __launch_bounds__(256, 3)
void lora_grad_kernel(GradJob ja, GradJob jb, int M) {
  const bool second = (int)blockIdx.x >= ja.tiles * ja.splits;
  const GradJob& j = second ? jb : ja;
  const int id = blockIdx.x - (second ? ja.tiles * ja.splits : 0);
  const int c0 = id % j.tiles * COLS, split = id / j.tiles;
  const int steps = (M + TILE - 1) / TILE;
  const int first = (int)((long)steps * split / j.splits);
  const int last = (int)((long)steps * (split + 1) / j.splits);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6), hi = lane >> 5;
  const int C = j.C, wide = min(COLS, C - c0);
  __shared__ __attribute__((aligned(16))) short zt[2][TILE * COLS], vt[2][TILE * RANK];

  auto stage = [&](int step, int buf) {
    const int m0 = step * TILE, left = M - m0;
    const short* src = j.z + (long)m0 * C + c0;
#pragma unroll
    for (int i = 0; i < TILE * COLS / 8; i += 256) {       // columns past the last: the first
      const int idx = i + tid, row = idx / (COLS / 8);
      const int c = ((idx % (COLS / 8)) ^ swz<COLS>(row)) * 8;
      load_to_lds16(src, (unsigned)(min(row, left - 1) * C + (c < wide ? c : 0)) * 2,
                    &zt[buf][(i + wid * 64) * 8]);
    }
    stage_tile<RANK>(j.v + (long)m0 * RANK, RANK, left, vt[buf]);
  };
  f32x16_t acc[2] = {f32x16_t{}, f32x16_t{}};
  if (first < last) stage(first, 0);
  for (int step = first, buf = 0; step < last; step++, buf ^= 1) {
    tiles_ready();
    if (step + 1 < last) stage(step + 1, buf ^ 1);
    const int left = M - step * TILE;
    if (left < TILE) {                                     // the last: no rows past the end
      for (int i = tid; i < (TILE - left) * COLS / 8; i += 256)
        *reinterpret_cast<s16x8*>(&zt[buf][left * COLS + i * 8]) = s16x8{};
      for (int i = tid; i < (TILE - left) * RANK / 8; i += 256)
        *reinterpret_cast<s16x8*>(&vt[buf][left * RANK + i * 8]) = s16x8{};
      __syncthreads();
    }
#pragma unroll
    for (int ks = 0; ks < TILE / 16; ks++) {
      const bf16x8 zf = col_frag<COLS>(zt[buf], 16 * ks, 32 * wid, lane);
#pragma unroll
      for (int t = 0; t < 2; t++)
        acc[t] = mfma32x32x16(zf, col_frag<RANK>(vt[buf], 16 * ks, 32 * t, lane), acc[t]);
    }
  }
  // lane: rank 32 t + lane % 32, columns c0 + 32 wid + crow(0 .. 15)
  float* part = j.splits > 1 ? j.part + (long)split * C * RANK : nullptr;
#pragma unroll
  for (int t = 0; t < 2; t++)
#pragma unroll
    for (int g = 0; g < 4; g++) {
      const int c = c0 + 32 * wid + crow(4 * g, hi), r = 32 * t + (lane & 31);
      if (c >= C) continue;                                // C is a multiple of 8
      float o[4];
#pragma unroll
      for (int k = 0; k < 4; k++) o[k] = acc[t][4 * g + k];
      if (j.flat) {
        if (part) stv<4>(part + (long)r * C + c, o);
        else stv<4>(j.out + (long)r * C + c, o);
      } else {
#pragma unroll
        for (int k = 0; k < 4; k++) {
          if (part) part[(long)(c + k) * RANK + r] = o[k];
          else j.out[(long)(c + k) * RANK + r] = f2bf(o[k]);
        }
      }
    }
}

// 4 elements per thread
__global__ __launch_bounds__(256)
void lora_grad_sum_kernel(GradJob ja, GradJob jb) {
  long i = ((long)blockIdx.x * 256 + threadIdx.x) * 4;
  const long na = ja.splits > 1 ? (long)ja.C * RANK : 0, nb = jb.splits > 1 ? (long)jb.C * RANK : 0;
  if (i >= na + nb) return;
  const GradJob& j = i < na ? ja : jb;
  if (i >= na) i -= na;
  const long n = (long)j.C * RANK;
  f32x4 s = *reinterpret_cast<const f32x4*>(j.part + i);
#pragma unroll 4
  for (int k = 1; k < j.splits; k++) s += *reinterpret_cast<const f32x4*>(j.part + k * n + i);
  float o[4] = {s[0], s[1], s[2], s[3]};
  stv<4>(j.out + i, o);
}

// (dA, dB) from x [M, K], du [M, 64], dy [M, N] and u [M, 64]; an empty tensor where
// x or dy is not given
std::vector<torch::Tensor> lora_grads(c10::optional<torch::Tensor> x,
                                      c10::optional<torch::Tensor> du,
                                      c10::optional<torch::Tensor> dy,
                                      c10::optional<torch::Tensor> u) {
  TORCH_CHECK(x || dy, "lora_grads: nothing to do");
  const long M = x ? x->size(0) : dy->size(0);
  const auto options = x ? x->options() : dy->options();
  on_gpu({x, du, dy, u});
  TORCH_CHECK(M > 0 && M < (1L << 31) - TILE, "lora_grads: tokens");
  std::vector<torch::Tensor> outs, keep;
  GradJob jobs[2] = {};
  long blocks = 0, sums = 0;
  for (int k = 0; k < 2; k++) {
    const auto& given = k ? dy : x;
    const auto& factor = k ? u : du;
    GradJob& j = jobs[k];
    j.splits = 1;
    if (!given) {
      outs.push_back(torch::empty({0}, options));
      continue;
    }
    TORCH_CHECK(factor.has_value(), "lora_grads: both factors");
    const long C = given->size(1);
    for (const auto& t : {*given, *factor})
      TORCH_CHECK(t.dim() == 2 && t.is_contiguous() && t.scalar_type() == torch::kBFloat16 &&
                  t.size(0) == M, "lora_grads: contiguous bf16 matrices");
    TORCH_CHECK(factor->size(1) == RANK && C % 8 == 0 && C > 0 && C < (1L << 24),
                "lora_grads: rank 64, columns a multiple of 8");
    const auto z = on16(*given), v = on16(*factor);
    keep.push_back(z);
    keep.push_back(v);
    j.flat = k == 0;
    outs.push_back(torch::empty({j.flat ? RANK : C, j.flat ? C : RANK}, options));
    j.z = (const short*)z.data_ptr();
    j.v = (const short*)v.data_ptr();
    j.out = (short*)outs.back().data_ptr();
    j.C = C;
    j.tiles = (C + COLS - 1) / COLS;
    // at most 512 workgroups, two for each CU, of at least 8 steps: 48720 tokens of 17920
    // columns 352 us in 3 parts (420 workgroups), 413 in 4; of 9728 193 in 6, 240 in 7
    const long steps = (M + TILE - 1) / TILE;
    j.splits = (int)std::max(1L, std::min<long>(512 / j.tiles, steps / 8));
    if (j.splits > 1) {
      keep.push_back(torch::empty({j.splits, C * RANK}, options.dtype(torch::kFloat32)));
      j.part = keep.back().data_ptr<float>();
      sums += C * RANK;
    }
    blocks += (long)j.tiles * j.splits;
  }
  auto stream = c10::hip::getCurrentHIPStream();
  hipLaunchKernelGGL(lora_grad_kernel, dim3(blocks), dim3(256), 0, stream, jobs[0], jobs[1],
                     (int)M);
  if (sums)
    hipLaunchKernelGGL(lora_grad_sum_kernel, dim3((sums / 4 + 255) / 256), dim3(256), 0, stream,
                       jobs[0], jobs[1]);
  HIP_CHECK_LAST();
  return outs;
}

// ------------------------------------------------------- down to the rank
// out [M, 64] = scale z p: p is A^T of A [64, C] (FLAT) or B [C, 64].  A workgroup
// owns 64 rows and a part of the columns, 64 at a time through three LDS buffers.
// Bound by reading z once; a few rows are divided among parts of the columns.  48720
// x 1536 37 us, library 38; 4096 x 8960 26, library 43; 240 x 896 7, library 14, and with
// the host's part 8.5 and 25.
template <bool FLAT>
__global__ __launch_bounds__(256, 3)
void lora_down_kernel(const short* __restrict__ z, const short* __restrict__ p,
                      short* __restrict__ out, float* __restrict__ parts, int M, int C, int splits,
                      float scale) {
  constexpr int R = 3, LOADS = 4;          // buffers, loads of a wave for one
  const int tile = blockIdx.x / splits, split = blockIdx.x % splits;
  const int m0 = tile * TILE, left = M - m0;
  const int steps = (C + TILE - 1) / TILE;
  const int first = (int)((long)steps * split / splits);
  const int last = (int)((long)steps * (split + 1) / splits);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6), hi = lane >> 5;
  const int rows0 = 32 * (wid & 1), rank0 = 32 * (wid >> 1);
  __shared__ __attribute__((aligned(16))) short zt[R][TILE * TILE], pt[R][TILE * RANK];

  const short* zb = z + (long)m0 * C;
  auto stage = [&](int step, int buf) {
    const int k0 = step * TILE, wide = min(TILE, C - k0);
#pragma unroll
    for (int i = 0; i < TILE * TILE / 8; i += 256) {       // columns past the last: the first
      const int idx = i + tid, row = idx >> 3, c = ((idx & 7) ^ swz<TILE>(row)) * 8;
      load_to_lds16(zb + k0, (unsigned)(min(row, left - 1) * C + (c < wide ? c : 0)) * 2,
                    &zt[buf][(i + wid * 64) * 8]);
    }
    if (FLAT) stage_tile<TILE>(p + k0, C, RANK, pt[buf]);
    else stage_tile<RANK>(p + (long)k0 * RANK, RANK, wide, pt[buf]);
  };
  f32x16_t acc{};
#pragma unroll
  for (int i = 0; i < R - 1; i++)
    if (first + i < last) stage(first + i, i);
  int buf = 0;
  for (int step = first; step < last; step++) {
    if (step + 1 < last) wait_loads<LOADS>();
    else wait_loads<0>();
    __syncthreads();
    if (step + R - 1 < last) stage(step + R - 1, buf + R - 1 >= R ? buf - 1 : buf + R - 1);
    const int wide = C - step * TILE;
    if (!FLAT && wide < TILE) {                            // the last: no columns past the end
      for (int i = tid; i < TILE * TILE / 8; i += 256) {
        const int row = i >> 3, c = ((i & 7) ^ swz<TILE>(row)) * 8;
        if (c >= wide) *reinterpret_cast<s16x8*>(&zt[buf][i * 8]) = s16x8{};
      }
      for (int i = tid; i < (TILE - wide) * RANK / 8; i += 256)
        *reinterpret_cast<s16x8*>(&pt[buf][wide * RANK + i * 8]) = s16x8{};
      __syncthreads();
    }
#pragma unroll
    for (int ks = 0; ks < TILE / 16; ks++) {
      const bf16x8 zf = row_frag<TILE>(zt[buf], rows0, ks, lane);
      const bf16x8 pf = FLAT ? row_frag<TILE>(pt[buf], rank0, ks, lane)
                             : col_frag<RANK, true>(pt[buf], 16 * ks, rank0, lane);
      acc = mfma32x32x16(pf, zf, acc);
    }
    buf = buf + 1 == R ? 0 : buf + 1;
  }
  // lane: row m0 + rows0 + lane % 32, ranks rank0 + crow(0 .. 15)
  const int m = m0 + rows0 + (lane & 31);
  if (m >= M) return;
#pragma unroll
  for (int g = 0; g < 4; g++) {
    const long at = (long)m * RANK + rank0 + crow(4 * g, hi);
    float o[4];
#pragma unroll
    for (int k = 0; k < 4; k++) o[k] = acc[4 * g + k] * scale;
    if (splits > 1) stv<4>(parts + (long)split * M * RANK + at, o);
    else stv<4>(out + at, o);
  }
}

__global__ __launch_bounds__(256)
void lora_down_sum_kernel(const float* __restrict__ parts, short* __restrict__ out, long n,
                          int splits) {
  const long i = ((long)blockIdx.x * 256 + threadIdx.x) * 4;
  if (i >= n) return;
  f32x4 s = *reinterpret_cast<const f32x4*>(parts + i);
#pragma unroll 4
  for (int k = 1; k < splits; k++) s += *reinterpret_cast<const f32x4*>(parts + k * n + i);
  float o[4] = {s[0], s[1], s[2], s[3]};
  stv<4>(out + i, o);
}

// scale z A^T with A [64, C], or scale z B with B [C, 64] (`flat` tells which)
torch::Tensor lora_down(torch::Tensor z, torch::Tensor p, double scale, bool flat) {
  on_gpu({z, p});
  for (const auto& t : {z, p})
    TORCH_CHECK(t.dim() == 2 && t.is_contiguous() && t.scalar_type() == torch::kBFloat16,
                "lora_down: contiguous bf16 matrices");
  const long M = z.size(0), C = z.size(1);
  TORCH_CHECK(p.size(flat ? 0 : 1) == RANK && p.size(flat ? 1 : 0) == C, "lora_down: rank 64");
  TORCH_CHECK(C > 0 && C % (flat ? TILE : 8) == 0 && C < (1L << 24) && M < (1L << 31) - TILE,
              "lora_down: columns a multiple of ", flat ? TILE : 8);
  auto out = torch::empty({M, RANK}, z.options());
  if (M == 0) return out;
  z = on16(z);
  p = on16(p);
  const long tiles = (M + TILE - 1) / TILE, steps = (C + TILE - 1) / TILE;
  // Parts of the columns that make it shortest, in us: a step of a workgroup takes 0.31
  // and the longer the more of them share the memory; a division costs another launch and
  // the parts' way through memory.
  // Measured in 1 / 2 / 4 parts: 240 x 1536 11.1 / 9.3 / 7.7, 4096 x 1536 11.4 / 10.5 / 10.6,
  // 8000 x 1536 11.7 / 12.1 / 12.7, 8000 x 8960 59 / 42 / 39, 16000 x 3584 32.4 / 31.8 / 34.4.
  int splits = 1;
  double best = 0;
  for (long n = 1; n <= std::min(16L, steps); n++) {
    const double us = (double)((steps + n - 1) / n) * std::max(0.31, 0.25 + (double)(tiles * n) * 0.0012) +
                      (n > 1 ? 2.2 + (double)(n * M) * 1e-4 : 0.0);
    if (n == 1 || us < best) {
      best = us;
      splits = (int)n;
    }
  }
  torch::Tensor parts;
  if (splits > 1) parts = torch::empty({splits, M * RANK}, z.options().dtype(torch::kFloat32));
  float* pp = splits > 1 ? parts.data_ptr<float>() : nullptr;
  auto stream = c10::hip::getCurrentHIPStream();
#define LAUNCH(FLAT)                                                                          \
  hipLaunchKernelGGL((lora_down_kernel<FLAT>), dim3(tiles * splits), dim3(256), 0, stream,    \
                     (const short*)z.data_ptr(), (const short*)p.data_ptr(),                  \
                     (short*)out.data_ptr(), pp, (int)M, (int)C, splits, (float)scale)
  if (flat) LAUNCH(true);
  else LAUNCH(false);
#undef LAUNCH
  if (splits > 1)
    hipLaunchKernelGGL(lora_down_sum_kernel, dim3((M * RANK / 4 + 255) / 256), dim3(256), 0,
                       stream, pp, (short*)out.data_ptr(), M * RANK, splits);
  HIP_CHECK_LAST();
  return out;
}
