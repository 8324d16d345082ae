// Linears of at most 64 rows (decoding): y = x w^T + bias, or the gated
// feed-forward's silu(x Wg^T) * (x Wu^T); and of more rows in blocks of 64, as far as all
// blocks fit the CUs at once.
//
// Bound by reading the weights and, with more than 16 rows, by fetching x into every
// CU.  The waves of a workgroup share the depth: each walks 64 elements at a time
// of its own part, which direct loads bring into a ring of its own in LDS, whole
// 128-byte lines, so that nothing waits at a barrier; at the end they add up
// through LDS.  (Fragments loaded straight into registers touch half a line at a
// time: 64 rows of 8960 x 1536, gated, 34 us.)  Deep products of few columns are
// also divided among workgroups, whose 32-bit parts rows_sum_kernel adds in order.
//
// us for 64 / 16 / 1 rows, library before -> now:
//   2048 x 1536       7.6 -> 6.8    7.1 -> 4.6    6.9 -> 4.1    (in two parts 5.2, 3.8, 3.6)
//   1536 x 8960       24.8 -> 10.7  27.9 -> 7.5   27.7 -> 7.2   (in five parts, without
//                                                               their sum: 4.6 by itself)
//   8960 x 1536, GLU  20.6 -> 16.4  41.6 -> 13.2  42.1 -> 13.0
//   151936 x 1536     115 -> 108    159 -> 90     158 -> 82     (467 MB: 5.7 TB/s)
// With 64 rows, the sums and stores of all tiles by one wave took as long as fetching x:
// 5.4, 11.8, 18.3 and 110 us.  Addresses made in the loads' own assembly, products between
// the loads, deeper rings and walks that start at different depths changed nothing.
#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>

#include "common.h"
#include "checks.h"

struct RowsArgs {
  const short *x, *w;      // [M, K], [N, K] (GLU: w2 the up weights)
  const short *w2, *bias;
  const short *u, *b;      // [M, 64], [N, 64]: an adapter's pair, the depth's last step
  short* y;                // [M, N]
  float* parts;            // [splits, M, N] instead of y
  int M, N, K;
};

// MF * 16 rows, NF * 16 weight rows; R chunks of 64 elements in each wave's ring.
// GLU: tiles of gate's and up's rows in turn, or (NF odd) 8 rows of each in a tile.
// BLOCKS: the grid's depth are blocks of so many rows; there are no parts.
template <int MF, int NF, int WAVES, int R, bool GLU, bool BLOCKS = false, bool LORA = false>
__global__ __launch_bounds__(WAVES * 64)
void linear_rows_kernel(RowsArgs a) {
  static_assert(BLOCKS || !LORA);
  if constexpr (BLOCKS) {
    const long m0 = (long)blockIdx.z * 16 * MF;
    a.x += m0 * a.K;
    if (LORA) a.u += m0 * 64;
    a.y += m0 * a.N;
    a.M = min(16 * MF, a.M - (int)m0);
  }
  constexpr int COLS = GLU ? NF * 8 : NF * 16;       // of y, of a workgroup
  constexpr bool HALVES = GLU && NF % 2;
  constexpr int CHUNK = (MF + NF) * 16 * 64, LOADS = (MF + NF) * 2;
  const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lo = lane & 15, hi = lane >> 4;
  const int n0 = blockIdx.x * COLS;
  __shared__ __attribute__((aligned(16))) short ring[WAVES][R][CHUNK];    // [w rows, x rows]

  // A load of a wave is 8 rows of 128 bytes, their 16-byte chunks exchanged (xor)
  // by row pair.
  unsigned wo[NF * 2], xo[MF * 2];
  const short* wb[GLU ? 2 : 1] = {a.w + (long)n0 * a.K};
  if (GLU) wb[GLU ? 1 : 0] = a.w2 + (long)n0 * a.K;
  auto spot = [&](int row, int most, int ld) {
    return (unsigned)(min(row, most) * ld + (((lane & 7) ^ ((lane >> 4) & 3)) << 3)) * 2;
  };
  auto spots = [&](int ld) {
#pragma unroll
    for (int i = 0; i < NF * 2; i++) {
      const int eight = HALVES ? i / 2 : GLU ? i / 4 * 2 + (i & 1) : i;
      wo[i] = spot(eight * 8 + (lane >> 3), a.N - 1 - n0, ld) ^ (i & 1) << 6;
    }
#pragma unroll
    for (int i = 0; i < MF * 2; i++)
      xo[i] = spot(8 * i + (lane >> 3), a.M - 1, ld) ^ (i & 1) << 6;
  };
  spots(a.K);
  // this wave's share of the depth
  const int deep = a.K / 64, steps = deep + LORA;
  const int shares = gridDim.y * WAVES, share = blockIdx.y * WAVES + wid;
  const int first = (int)((long)steps * share / shares);
  const int last = (int)((long)steps * (share + 1) / shares);
  const short* xb = a.x;
  auto fetch = [&](int step, int slot) {
    int k0 = step * 64;
    short* at = ring[wid][slot];
    if (LORA && step == deep) {       // the last that its wave asks for
      spots(64);
      xb = a.u;
      wb[0] = a.b + (long)n0 * 64;
      k0 = 0;
    }
#pragma unroll
    for (int i = 0; i < NF * 2; i++)
      load_to_lds16(wb[GLU ? (HALVES ? i : i / 2) & 1 : 0] + k0, wo[i], at + i * 512);
#pragma unroll
    for (int i = 0; i < MF * 2; i++) load_to_lds16(xb + k0, xo[i], at + (NF * 2 + i) * 512);
  };

  f32x4 acc[NF][MF];
#pragma unroll
  for (int i = 0; i < NF; i++)
#pragma unroll
    for (int j = 0; j < MF; j++) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < R; i++)
    if (first + i < last) fetch(first + i, i);
  int slot = 0;
  for (int step = first; step < last; step++) {
    chunk_ready<LOADS, R>(last - 1 - step);
    const short* at = ring[wid][slot];
    auto part = [&](int row16, int q) {
      return frag(at + (row16 * 16 + lo) * 64 + (((4 * q + hi) ^ ((lo >> 1) & 7)) << 3));
    };
    bf16x8l wf[2][NF], xf[2][MF];
#pragma unroll
    for (int q = 0; q < 2; q++) {
#pragma unroll
      for (int i = 0; i < NF; i++) wf[q][i] = part(i, q);
#pragma unroll
      for (int j = 0; j < MF; j++) xf[q][j] = part(NF + j, q);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");       // read before it is filled again
    if (step + R < last) fetch(step + R, slot);
    slot = slot + 1 == R ? 0 : slot + 1;
#pragma unroll
    for (int q = 0; q < 2; q++)
#pragma unroll
      for (int i = 0; i < NF; i++)
#pragma unroll
        for (int j = 0; j < MF; j++) acc[i][j] = mfma16l(wf[q][i], xf[q][j], acc[i][j]);
  }
  __syncthreads();
  // Each wave adds up and stores its share of the tiles, always in the same order, so that
  // one barrier is all and no wave is left with the stores of all: with 64 rows that
  // took longer than fetching x.  A unit is a tile, or a gate's and its up's.
  constexpr int TILES = GLU && !HALVES ? 2 : 1, UNITS = NF / TILES * MF;
  typedef f32x4 Tile[64];
  static_assert(sizeof(Tile) * UNITS * TILES * (WAVES - 1) <= sizeof(ring), "room for the sums");
  Tile* sums = reinterpret_cast<Tile*>(&ring[0][0][0]);
#pragma unroll
  for (int u = 0; u < UNITS; u++) {
    const int owner = u % WAVES;
    if (wid == owner) continue;
#pragma unroll
    for (int e = 0; e < TILES; e++)
      sums[(u * TILES + e) * (WAVES - 1) + wid - (wid > owner)][lane] =
          acc[u / MF * TILES + e][u % MF];
  }
  __syncthreads();
  // lane: row 16 j + lo, columns 16 i + 4 hi .. + 3 (HALVES: 8 i + 4 hi .. + 3, up's
  // in the wave's upper half)
  const bool whole = a.N % 4 == 0;
#pragma unroll
  for (int u = 0; u < UNITS; u++) {
    const int owner = u % WAVES, i = u / MF * TILES, j = u % MF;
    if (wid != owner) continue;
    f32x4 sum[TILES];
#pragma unroll
    for (int e = 0; e < TILES; e++) {
      f32x4 w[WAVES];
#pragma unroll
      for (int k = 0; k < WAVES; k++)
        w[k] = k == owner ? acc[i + e][j]
                          : sums[(u * TILES + e) * (WAVES - 1) + k - (k > owner)][lane];
#pragma unroll
      for (int n = WAVES / 2; n > 0; n >>= 1)
#pragma unroll
        for (int k = 0; k < n; k++) w[k] += w[k + n];
      sum[e] = w[0];
    }
    const int m = 16 * j + lo, n = n0 + (GLU ? i * 8 : i * 16) + 4 * hi;
    float v[4];
#pragma unroll
    for (int r = 0; r < 4; r++) {
      v[r] = sum[0][r];
      if (GLU)
        v[r] = silu_fast(v[r]) * (HALVES ? __shfl_xor(v[r], 32) : sum[TILES - 1][r]);
      else if (a.bias && n + r < a.N)
        v[r] += bf2f(a.bias[n + r]);
    }
    if (m >= a.M || (HALVES && hi > 1)) continue;
    if (!BLOCKS && a.parts) {
      float* p = a.parts + ((long)blockIdx.y * a.M + m) * a.N + n;
      if (whole && n < a.N) stv<4>(p, v);
      else
        for (int r = 0; r < 4; r++)
          if (n + r < a.N) p[r] = v[r];
    } else {
      short* p = a.y + (long)m * a.N + n;
      if (whole && n < a.N) stv<4>(p, v);
      else
        for (int r = 0; r < 4; r++)
          if (n + r < a.N) stf(p + r, v[r]);
    }
  }
}

__global__ __launch_bounds__(256)
void rows_sum_kernel(const float* __restrict__ parts, const short* __restrict__ bias,
                     short* __restrict__ y, long n, int N, int splits) {
  const long i = ((long)blockIdx.x * 256 + threadIdx.x) * 4;
  if (i >= n) return;
  f32x4 s = *reinterpret_cast<const f32x4*>(parts + i);
  for (int k = 1; k < splits; k++) s += *reinterpret_cast<const f32x4*>(parts + k * n + i);
  float v[4];
#pragma unroll
  for (int r = 0; r < 4; r++) v[r] = s[r] + (bias ? bf2f(bias[(i + r) % N]) : 0.f);
  stv<4>(y + i, v);
}

static void check_rows(const torch::Tensor& x, const torch::Tensor& w, long most = 64) {
  for (const auto& t : {x, w})
    TORCH_CHECK(t.dim() == 2 && t.is_contiguous() && t.scalar_type() == torch::kBFloat16 &&
                (uintptr_t)t.data_ptr() % 16 == 0, "linear_rows: contiguous bf16 matrices");
  // a workgroup's offsets, of up to 128 rows, are 32-bit bytes
  TORCH_CHECK(x.size(0) <= most && x.size(1) == w.size(1) && x.size(1) % 64 == 0 &&
              x.size(1) < (1L << 24) && w.size(0) < (1L << 30),
              "linear_rows: at most ", most, " rows, depth a multiple of 64 below 2^24");
}

template <int NF, int WAVES, int R, bool GLU>
static void launch_rows(const RowsArgs& a, int splits) {
  constexpr int COLS = GLU ? NF * 8 : NF * 16;
  const dim3 grid((a.N + COLS - 1) / COLS, splits);
#define LAUNCH(MF)                                                                           \
  hipLaunchKernelGGL((linear_rows_kernel<MF, NF, WAVES, R, GLU>), grid, dim3(WAVES * 64), 0, \
                     c10::hip::getCurrentHIPStream(), a)
  switch ((a.M + 15) / 16) {
    case 1: LAUNCH(1); break;
    case 2: LAUNCH(2); break;
    case 3: LAUNCH(3); break;
    default: LAUNCH(4);
  }
#undef LAUNCH
}

// y [M, N], or with `deferred`, where the depth is divided, its 32-bit parts [splits, M, N],
// which the next kernel adds up
static torch::Tensor rows_product(torch::Tensor x, torch::Tensor w,
                                  c10::optional<torch::Tensor> bias, bool deferred) {
  on_gpu({x, w, bias});
  check_rows(x, w);
  const long M = x.size(0), K = x.size(1), N = w.size(0);
  if (bias)
    TORCH_CHECK(bias->scalar_type() == torch::kBFloat16 && bias->is_contiguous() &&
                bias->numel() == N, "linear_rows: bf16 bias");
  if (M == 0 || N == 0) return torch::empty({M, N}, x.options());
  RowsArgs a{};
  a.x = (const short*)x.data_ptr();
  a.w = (const short*)w.data_ptr();
  const short* b = bias ? (const short*)bias->data_ptr() : nullptr;
  a.M = M;
  a.N = N;
  a.K = K;
  // 16 columns each while that makes at most a workgroup per CU, since the rows of
  // x are read by each; up to 64 for more columns, 96 and four waves for the widest
  // with more than 32 rows, where that shares x better: 64 rows of 151936 x 1536 108 us, 113
  // with 64 and two, of x 896 65.8 and 71.7; 32 rows 97.6 and 95.6.  A deep product of few columns is divided until about
  // 224 workgroups share it, which has to pay for a second kernel of 3 us: 64 rows of
  // 1536 x 8960 15 us in 4 parts, 24 in one; 1536 x 1536 6 us in one, 7 in 2.  Without
  // that kernel a shallow one is divided by two where it leaves half of the CUs idle: 64 rows
  // of 2048 x 1536 7.1 us, 5.4 in 2 parts, 16 rows 4.6 and 3.9, one 4.1 and 3.7; 64 of 896 x
  // 896 4.6 and 3.9.  A deep one
  // of many columns wants many waves in flight on each: one row of 14336 x 4096 24 us
  // with 32 columns and four waves, 32 with 64 and two.
  const bool deep = K > 2048, shared = deep && N <= 5120;
  const int nf = shared ? (N <= 1024 ? 1 : N < 3200 ? 2 : 4)
                 : deep ? 2 : N <= 4096 ? 1 : N <= 8192 ? 2 : 4;
  const long tiles = (N + 16 * nf - 1) / (16 * nf);
  int splits = 1;
  if (N % 4 == 0 && shared) splits = (int)std::min(8L, std::max(1L, (224 + tiles / 2) / tiles));
  else if (N % 4 == 0 && deferred && !deep && tiles <= 128 && K >= 512) splits = 2;
  torch::Tensor y, parts;
  if (splits > 1) {
    parts = torch::empty({splits, M, N}, x.options().dtype(torch::kFloat32));
    a.parts = parts.data_ptr<float>();
  } else {
    a.bias = b;
  }
  if (splits == 1 || !deferred) {
    y = torch::empty({M, N}, x.options());
    a.y = (short*)y.data_ptr();
  }
  if (nf == 1) launch_rows<1, 4, 3, false>(a, splits);
  else if (nf == 2) launch_rows<2, 4, 3, false>(a, splits);
  else if (M <= 32 || N <= 65536) launch_rows<4, 2, 2, false>(a, splits);
  else launch_rows<6, 4, 1, false>(a, splits);
  if (splits > 1 && !deferred)
    hipLaunchKernelGGL(rows_sum_kernel, dim3((M * N / 4 + 255) / 256), dim3(256), 0,
                       c10::hip::getCurrentHIPStream(), a.parts, b, a.y, M * N, (int)N, splits);
  HIP_CHECK_LAST();
  return y.defined() ? y : parts;
}

torch::Tensor linear_rows(torch::Tensor x, torch::Tensor w, c10::optional<torch::Tensor> bias) {
  return rows_product(x, w, bias, false);
}

bool linear_blocks_fill(long M, long N) { return (M + 63) / 64 * ((N + 63) / 64) <= 256; }

template <bool LORA>
static void launch_blocks(const RowsArgs& a) {
  const int blocks = (a.M + 63) / 64;
#define LAUNCH(NF, R)                                                                         \
  hipLaunchKernelGGL((linear_rows_kernel<4, NF, 4, R, false, true, LORA>),                    \
                     dim3((a.N + 16 * NF - 1) / (16 * NF), 1, blocks), dim3(256), 0,          \
                     c10::hip::getCurrentHIPStream(), a)
  // as few columns to a workgroup as leave one a CU: rows are read again by each
  if ((long)blocks * ((a.N + 15) / 16) <= 256) LAUNCH(1, 3);
  else if ((long)blocks * ((a.N + 31) / 32) <= 256) LAUNCH(2, 3);
  else LAUNCH(4, 2);
#undef LAUNCH
  HIP_CHECK_LAST();
}

// x w^T + bias of any number of rows in blocks of 64.  Bound by latencies and by each workgroup's fetch of its rows and columns: 212 rows of
// 1536 x 1536 6.2 us (library 7.7), 640 8.7 (9.0), 212 of 896 x 4864 9.3 (11.8); a call is 4
// to 5 us of the host's time, a library call 19 to 22.
torch::Tensor linear_blocks(torch::Tensor x, torch::Tensor w, c10::optional<torch::Tensor> bias) {
  on_gpu({x, w, bias});
  check_rows(x, w, 1L << 24);
  TORCH_CHECK(!bias || (bias->scalar_type() == torch::kBFloat16 && bias->is_contiguous() &&
                        bias->numel() == w.size(0)), "linear_blocks: bf16 bias");
  auto y = torch::empty({x.size(0), w.size(0)}, x.options());
  if (y.numel() == 0) return y;
  RowsArgs a{};
  a.x = (const short*)x.data_ptr();
  a.w = (const short*)w.data_ptr();
  a.bias = bias ? (const short*)bias->data_ptr() : nullptr;
  a.y = (short*)y.data_ptr();
  a.M = x.size(0);
  a.N = w.size(0);
  a.K = x.size(1);
  launch_blocks<false>(a);
  return y;
}

// the same with an adapter: x w^T + u b^T + bias
torch::Tensor lora_blocks(torch::Tensor x, torch::Tensor w, torch::Tensor u, torch::Tensor b,
                          c10::optional<torch::Tensor> bias) {
  check_rows(x, w, 1L << 24);
  check_rows(u, b, 1L << 24);
  TORCH_CHECK(u.size(1) == 64 && u.size(0) == x.size(0) && b.size(0) == w.size(0),
              "lora_blocks: an adapter of 64");
  TORCH_CHECK(!bias || (bias->scalar_type() == torch::kBFloat16 && bias->is_contiguous() &&
                        bias->numel() == w.size(0)), "lora_blocks: bf16 bias");
  auto y = torch::empty({x.size(0), w.size(0)}, x.options());
  RowsArgs a{};
  a.x = (const short*)x.data_ptr();
  a.w = (const short*)w.data_ptr();
  a.u = (const short*)u.data_ptr();
  a.b = (const short*)b.data_ptr();
  a.bias = bias ? (const short*)bias->data_ptr() : nullptr;
  a.y = (short*)y.data_ptr();
  a.M = x.size(0);
  a.N = w.size(0);
  a.K = x.size(1);
  launch_blocks<true>(a);
  return y;
}

// x w^T + bias as bf16 [M, N], or float32 [parts, M, N] that add up to x w^T alone
torch::Tensor linear_rows_parts(torch::Tensor x, torch::Tensor w,
                                c10::optional<torch::Tensor> bias) {
  return rows_product(x, w, bias, true);
}

// silu(x gate^T) * (x up^T)
torch::Tensor glu_rows(torch::Tensor x, torch::Tensor gate, torch::Tensor up) {
  on_gpu({x, gate, up});
  check_rows(x, gate);
  check_rows(x, up);
  TORCH_CHECK(gate.sizes() == up.sizes(), "glu_rows: gate and up alike");
  const long M = x.size(0), N = gate.size(0);
  auto y = torch::empty({M, N}, x.options());
  if (M == 0 || N == 0) return y;
  RowsArgs a{};
  a.x = (const short*)x.data_ptr();
  a.w = (const short*)gate.data_ptr();
  a.w2 = (const short*)up.data_ptr();
  a.y = (short*)y.data_ptr();
  a.M = M;
  a.N = N;
  a.K = x.size(1);
  // Of 16, 32, 40 and 48 columns to a workgroup those with which the 256 CUs, one workgroup
  // each, are through soonest, more rather than fewer where it makes no difference: 64 rows
  // of 7168 x 2048 16 us with 32, 20 with 40; 8960 x 1536 18.6 with 40, 25 with 16; 11008 x
  // 2048 22 with 48, 31 with 40 (276 workgroups); 18944 x 3584 58 with 40, 61 and 80 with
  // 48 and 32.
  long best = 0, cost = 0;
  for (long cols : {48L, 40L, 32L, 16L}) {
    const long c = ((N + cols - 1) / cols + 255) / 256 * cols;
    if (!best || c < cost) {
      best = cols;
      cost = c;
    }
  }
  if (best == 16) launch_rows<2, 2, 3, true>(a, 1);
  // twice the waves where there is as much to do for each: 64 rows of 8960 x 1536 16.4 us, 18.4
  // with two, 48 of 18944 x 3584 53.8 and 52.2; with 32 columns 64 rows of 14336 x 4096 50.6 and
  // 55.2, one to 16 41 and 50, 64 of 7168 x 2048 15.9 and 15.1
  else if (best == 32 && a.K > 2048) launch_rows<4, 4, 2, true>(a, 1);
  else if (best == 32) launch_rows<4, 2, 2, true>(a, 1);
  else if (best == 40 && M > 48) launch_rows<5, 4, 2, true>(a, 1);
  else if (best == 40) launch_rows<5, 2, 2, true>(a, 1);
  else launch_rows<6, 2, 2, true>(a, 1);
  HIP_CHECK_LAST();
  return y;
}
