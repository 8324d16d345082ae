// bf16 products of many rows, y = x w^T, in tiles of 256 x 256: with an adapter's
// rank-64 pair as one more step of the depth and a bias (lora.hip), or of a gated
// feed-forward's two weights at once, whose columns meet before they are rounded
// (glu.hip).
#pragma once

#include <hip/hip_runtime.h>

#include "common.h"

// ---- 256 x 256 tile, 8 waves -----------------------------------------------
// For grids that fill most of the chip with one workgroup per CU.  Twice the
// reuse of the 128-tile in both directions, LDS tiles without bank conflicts, the
// next step's fragments read between the products, 16 neighbouring columns of y
// per lane.  48720 x 17920 x 1536 + 64: 2.65 ms (1056 TFLOP/s) against 3.80, x 1536
// x 17920: 2.36 (1142) against 3.30; 59% of the cycles are products, the rest
// mostly waits at the tiles' barriers.  Four stages of 32 that land a barrier
// ahead (974 TFLOP/s: rows of 64 bytes double the requests), 256 x 128 tiles twice
// per CU (870) and four waves of 128 x 128 (999) were slower.
typedef __bf16 bf16x8_m __attribute__((ext_vector_type(8)));

constexpr int BIG = 256;

// 16-byte chunk exchange (xor) of a tile row: rows are 128 bytes apart, so two
// fill the banks.  Fragments take 16 rows in order from x, and from w rows
// 0-3, 16-19, 4-7, 20-23 (see wrow).
DEVINL int xswz(int row) { return (row >> 1) & 7; }
DEVINL int wswz(int row) { return ((row >> 1) & 3) | ((row >> 4) & 1) << 2; }
// the MFMA's row i of 32 is y's column wrow(i): a lane then holds 16 neighbours
DEVINL int wrow(int i) { return 16 * ((i >> 2) & 1) + (i & 3) + 4 * (i >> 3); }

// ACT: a tile has 128 columns of y; of every 64 rows of its w tile the first half is
// w's and the second the same columns of w2, and y = act(x w) * (x w2).
enum { NO_ACT, SILU_GLU, GELU_GLU };

template <int ACT>
DEVINL float glu(float g, float up) {
  const float z = ACT == SILU_GLU ? g : 1.5957691216057308f * (g + 0.044715f * g * g * g);
  return g * __builtin_amdgcn_rcpf(1.f + __expf(-z)) * up;      // gelu_tanh: x sigmoid(2 ..)
}

template <bool HAS_LORA, bool HAS_BIAS, bool VEC, int ACT>
__global__ __launch_bounds__(512, 2)
void gemm_big_kernel(const short* __restrict__ x, const short* __restrict__ w,
                     const short* __restrict__ u, const short* __restrict__ b,
                     const float* __restrict__ bias, const short* __restrict__ w2,
                     short* __restrict__ y, long ldy, int M, int N, int K1, int grid_m,
                     int grid_n) {
  constexpr int TN = ACT ? BIG / 2 : BIG;
  __shared__ __attribute__((aligned(16))) short lds[2][2][BIG * 64];   // [buffer][x, w]
  int wg = blockIdx.x;
  {
    const int nwg = gridDim.x, q = nwg >> 3, r = nwg & 7;
    const int xcd = wg & 7, i = wg >> 3;
    wg = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + i;
  }
  constexpr int GM = 8;       // tiles that run together share rows and columns
  const int group = wg / (GM * grid_n), first = group * GM;
  const int rows_here = min(GM, grid_m - first);
  const int bm = first + (wg - group * GM * grid_n) % rows_here;
  const int bn = (wg - group * GM * grid_n) / rows_here;
  const int m0 = bm * BIG, n0 = bn * TN;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = (wid >> 2) * 128, wn = (wid & 3) * 64;
  const int lo = lane & 31, hi = lane >> 5;
  const int n_k1 = K1 >> 6, n_kt = n_k1 + (HAS_LORA ? 1 : 0);

  // thread's rows of a tile: tid / 8 + 64 i; its chunk of each the same
  unsigned xo[4], wo[4];
  auto offsets = [&](int ld) {
    const int r = tid >> 3;
#pragma unroll
    for (int i = 0; i < 4; i++) {
      xo[i] = (unsigned)(min(r + 64 * i, M - 1 - m0) * ld + (((tid & 7) ^ xswz(r)) << 3)) * 2;
      const int n = ACT ? (r & 31) + 32 * i : r + 64 * i;
      wo[i] = (unsigned)(min(n, N - 1 - n0) * ld + (((tid & 7) ^ wswz(r)) << 3)) * 2;
    }
  };
  offsets(K1);
  const short *xb = x + (long)m0 * K1, *wb = (ACT && wid >= 4 ? w2 : w) + (long)n0 * K1;
  auto stage = [&](int kt, int buf) {
    const short *xs = xb + kt * 64, *ws = wb + kt * 64;
    if (HAS_LORA && kt == n_k1) {
      offsets(64);
      xs = u + (long)m0 * 64;
      ws = b + (long)n0 * 64;
    }
#pragma unroll
    for (int i = 0; i < 4; i++) load_to_lds16(xs, xo[i], &lds[buf][0][(i * 512 + wid * 64) * 8]);
#pragma unroll
    for (int i = 0; i < 4; i++) load_to_lds16(ws, wo[i], &lds[buf][1][(i * 512 + wid * 64) * 8]);
  };
  const int xr = wm + lo, wr = wn + wrow(lo);
  auto xfrag = [&](int buf, int mt, int ks) {
    return *reinterpret_cast<const bf16x8_m*>(
        &lds[buf][0][(xr + 32 * mt) * 64 + (((2 * ks + hi) ^ xswz(xr)) << 3)]);
  };
  auto wfrag = [&](int buf, int nt, int ks) {
    return *reinterpret_cast<const bf16x8_m*>(
        &lds[buf][1][(wr + 32 * nt) * 64 + (((2 * ks + hi) ^ wswz(wr)) << 3)]);
  };

  f32x16 acc[4][2];
#pragma unroll
  for (int i = 0; i < 4; i++)
#pragma unroll
    for (int j = 0; j < 2; j++) acc[i][j] = f32x16{};

  stage(0, 0);
  for (int kt = 0; kt < n_kt; kt++) {
    const int buf = kt & 1;
    wait_loads<0>();
    __syncthreads();
    bf16x8_m xf[2][4], wf[2][2];
    auto read = [&](int ks) {
#pragma unroll
      for (int j = 0; j < 2; j++) wf[ks & 1][j] = wfrag(buf, j, ks);
#pragma unroll
      for (int i = 0; i < 4; i++) xf[ks & 1][i] = xfrag(buf, i, ks);
    };
    read(0);
    if (kt + 1 < n_kt) stage(kt + 1, buf ^ 1);
    // the next step's fragments are read between this one's products
#pragma unroll
    for (int ks = 0; ks < 4; ks++) {
      if (ks < 3) read(ks + 1);
#pragma unroll
      for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < 2; j++)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wf[ks & 1][j], xf[ks & 1][i],
                                                              acc[i][j], 0, 0, 0);
#pragma unroll
      for (int g = 0; g < 6; g++) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);      // product
        if (ks < 3) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);      // LDS read
      }
      __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
    }
  }
  // lane: row m0 + wm + 32 i + lo, columns n0 + wn + 32 j + 16 hi + 0..15
#pragma unroll
  for (int j = 0; j < (ACT ? 1 : 2); j++) {
    const int gn = n0 + (ACT ? wn / 2 : wn + 32 * j) + 16 * hi;
    float bv[16];
    if (HAS_BIAS) {
#pragma unroll
      for (int r = 0; r < 16; r++) bv[r] = bias[min(gn + r, N - 1)];
    }
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int gm = m0 + wm + 32 * i + lo;
      if (gm >= M) continue;
      short* dst = y + gm * ldy + gn;
#pragma unroll
      for (int h = 0; h < 2; h++) {
        s16x8 o;
#pragma unroll
        for (int r = 0; r < 8; r++)
          o[r] = f2bf(ACT ? glu<ACT>(acc[i][0][8 * h + r], acc[i][1][8 * h + r])
                          : acc[i][j][8 * h + r] + (HAS_BIAS ? bv[8 * h + r] : 0.f));
        if (VEC) {
          if (gn + 8 * h < N) *reinterpret_cast<s16x8*>(dst + 8 * h) = o;
        } else {
#pragma unroll
          for (int r = 0; r < 8; r++)
            if (gn + 8 * h + r < N) dst[8 * h + r] = o[r];
        }
      }
    }
  }
}
