// Mixture of experts and linears per group.
//
// moe_route: 32-bit router logits, the top choices and their softmax, then for
// every expert the list of the rows (token * top + choice) that use it, in
// order.  Lists have room for every token, so nothing downstream waits for the
// counts.
//
// Grouped products: group g multiplies its rows (gathered through its list, or
// all rows at an offset of their own per group) by its own weights [N][K].  A
// workgroup finds its group and rows from the counts, so the grid is made for
// the worst case and surplus workgroups leave at once.
//   big      gemm_big.h's kernel of 256 x 256 tiles: groups of many rows
//   tiles    bf16 MFMA, 128 x 128 tiles through LDS: fewer, or sizes that are not its
//   stream   bf16 MFMA, 16, 32 or 64 rows, every wave by itself through a ring in LDS:
//            groups of few rows, bound by reading the weights
//   plain    scalar products in 32-bit, any type and any size
#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>

#include "common.h"
#include "checks.h"
#include "gemm_big.h"

struct Grouped {
  const void *a, *w;
  void* out;
  long lda, ga;          // row stride of a, its offset per group
  long ldw, gw, up;      // row and group stride of w; from gate to up weights
  long ldo, go;
  const int* lists;      // [G, cap] rows of each group, or null: 0 .. rows - 1
  const int* counts;     // [G]
  const float* scale;    // by row, or null
  int rows, cap, div;    // a row of a is list entry / div
  int G, N, K;
};

// group, first row and number of rows of row-tile `tile`; the same for a wave
DEVINL bool find_rows(const Grouped& a, int tile, int BM, int& g, int& m0, int& rows) {
  if (!a.lists) {
    const int per = (a.rows + BM - 1) / BM;
    g = tile / per;
    m0 = (tile % per) * BM;
    rows = a.rows;
    return g < a.G;
  }
  const int lane = threadIdx.x & 63;
  int before = 0;
  for (int base = 0; base < a.G; base += 64) {
    const int c = base + lane < a.G ? a.counts[base + lane] : 0;
    const int t = (c + BM - 1) / BM;
    int s = t;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int y = __shfl_up(s, off);
      if (lane >= off) s += y;
    }
    const int total = __shfl(s, 63);
    if (tile < before + total) {
      const int l = __ffsll((unsigned long long)__ballot(before + s > tile)) - 1;
      g = base + l;
      m0 = (tile - before - __shfl(s - t, l)) * BM;
      rows = __shfl(c, l);
      return true;
    }
    before += total;
  }
  return false;
}

// ------------------------------------------------------ plain, any type
// 64 x 64 tile, 4 x 4 per thread.  GLU: out = silu(gate) * up.
template <typename T, bool GLU>
__global__ __launch_bounds__(256) void grouped_plain_kernel(Grouped a) {
  constexpr int BK = 16, NB = GLU ? 2 : 1;
  __shared__ float as[BK][68], ws[NB][BK][68];
  int g, m0, rows;
  if (!find_rows(a, blockIdx.y, 64, g, m0, rows)) return;
  const int n0 = blockIdx.x * 64;
  const int* list = a.lists ? a.lists + (long)g * a.cap : nullptr;
  const T* A = (const T*)a.a + g * a.ga;
  const T* W = (const T*)a.w + g * a.gw;
  const int tm = threadIdx.x >> 4, tn = threadIdx.x & 15;
  float acc[NB][4][4] = {};
  for (int k0 = 0; k0 < a.K; k0 += BK) {
    for (int i = threadIdx.x; i < 64 * BK; i += 256) {
      const int m = i / BK, k = i % BK;
      float x = 0.f;
      if (m0 + m < rows && k0 + k < a.K) {
        const int id = list ? list[m0 + m] : m0 + m;
        x = ldf(A + (long)(id / a.div) * a.lda + k0 + k);
      }
      as[k][m] = x;
#pragma unroll
      for (int b = 0; b < NB; b++)
        ws[b][k][m] = (n0 + m < a.N && k0 + k < a.K)
                          ? ldf(W + b * a.up + (long)(n0 + m) * a.ldw + k0 + k) : 0.f;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < BK; k++)
#pragma unroll
      for (int b = 0; b < NB; b++)
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
          for (int j = 0; j < 4; j++) acc[b][i][j] += as[k][4 * tm + i] * ws[b][k][4 * tn + j];
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const int m = m0 + 4 * tm + i;
    if (m >= rows) continue;
    const int id = list ? list[m] : m;
    const float sc = a.scale ? a.scale[id] : 1.f;
    T* o = (T*)a.out + g * a.go + (long)id * a.ldo;
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const int n = n0 + 4 * tn + j;
      if (n >= a.N) continue;
      const float x = GLU ? act_silu(acc[0][i][j]) * acc[NB - 1][i][j] : acc[0][i][j];
      stf(o + n, x * sc);
    }
  }
}

// ---------------------------------------------------------- bf16 matrix cores
// The weights are the first operand, so a lane ends up with four neighbouring
// columns of one row.  GLU: every other 16 weight rows of a tile are up's, the
// ones between gate's of the same columns.
#define GLDS16(gsrc, ldst)                                   \
  __builtin_amdgcn_global_load_lds(                          \
      (const __attribute__((address_space(1))) void*)(gsrc), \
      (__attribute__((address_space(3))) void*)(ldst), 16, 0, 0)

__device__ __attribute__((aligned(16))) const short zero_chunk[8] = {};

template <bool GLU>
DEVINL const short* weight_row(const Grouped& a, const short* W, int n0, int r) {
  const int n = GLU ? n0 + (r >> 5) * 16 + (r & 15) : n0 + r;
  return W + (GLU && (r & 16) ? a.up : 0) + (long)min(n, a.N - 1) * a.ldw;
}

template <bool GLU>
DEVINL void store_row(const Grouped& a, short* o, int n, const f32x4& x, const f32x4& y, float sc,
                      bool wide) {
  float v[4];
#pragma unroll
  for (int j = 0; j < 4; j++) v[j] = (GLU ? act_silu(x[j]) * y[j] : x[j]) * sc;
  if (wide && n + 4 <= a.N) {
    stv<4>(o + n, v);
  } else {
#pragma unroll
    for (int j = 0; j < 4; j++)
      if (n + j < a.N) stf(o + n + j, v[j]);
  }
}

// 128 rows by 128 weight rows, 64 deep, two buffers filled straight from memory;
// four waves of 64 x 64.  The 16-byte chunks of an LDS row are exchanged (xor) by
// row, on the way in by choosing what each lane fetches.
template <bool GLU>
__global__ __launch_bounds__(256, 2) void grouped_tiles_kernel(Grouped a, int tiles_m,
                                                               int tiles_n) {
  __shared__ __attribute__((aligned(16))) short lds[2][2][128 * 64];
  // neighbours in one chiplet's L2: 8 row-tiles of each column-tile in turn
  int wg = blockIdx.x;
  {
    const int nwg = gridDim.x, q = nwg >> 3, r = nwg & 7, xcd = wg & 7, i = wg >> 3;
    wg = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + i;
  }
  const int per = 8 * tiles_n, first = wg / per * 8, rest = wg % per;
  const int wide8 = min(8, tiles_m - first);
  const int tm = first + rest % wide8, tn = rest / wide8;
  int g, m0, rows;
  if (!find_rows(a, tm, 128, g, m0, rows)) return;
  const int n0 = tn * (GLU ? 64 : 128);
  const int* list = a.lists ? a.lists + (long)g * a.cap : nullptr;
  const short* A = (const short*)a.a + g * a.ga;
  const short* W = (const short*)a.w + g * a.gw;
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const int wm = wid >> 1, wn = wid & 1, lo = lane & 15, hi = lane >> 4;

  const int wave0 = __builtin_amdgcn_readfirstlane(tid & ~63);
  const short *ap[4], *wp[4];              // this lane's chunks of a tile
  int kc[4];
#pragma unroll
  for (int x = 0; x < 4; x++) {
    const int c = x * 256 + tid, row = c >> 3;
    kc[x] = ((c & 7) ^ (row & 7)) * 8;
    const int i = min(m0 + row, rows - 1);
    ap[x] = A + (long)((list ? list[i] : i) / a.div) * a.lda + kc[x];
    wp[x] = weight_row<GLU>(a, W, n0, row) + kc[x];
  }
  auto stage = [&](int kt, int buf) {
    const int k0 = kt * 64;
#pragma unroll
    for (int x = 0; x < 4; x++) {
      const bool in = k0 + kc[x] < a.K;
      GLDS16(in ? ap[x] + k0 : zero_chunk, &lds[buf][0][(x * 256 + wave0) * 8]);
      GLDS16(in ? wp[x] + k0 : zero_chunk, &lds[buf][1][(x * 256 + wave0) * 8]);
    }
  };

  f32x4 acc[4][4];                         // [weight rows][rows]
#pragma unroll
  for (int i = 0; i < 4; i++)
#pragma unroll
    for (int j = 0; j < 4; j++) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int nk = (a.K + 63) / 64;
  stage(0, 0);
  __syncthreads();
  for (int kt = 0; kt < nk; kt++) {
    const int buf = kt & 1;
    if (kt + 1 < nk) stage(kt + 1, buf ^ 1);
#pragma unroll
    for (int kk = 0; kk < 2; kk++) {
      const int ch = ((kk * 4 + hi) ^ (lo & 7)) * 8;
      bf16x8l af[4], wf[4];
#pragma unroll
      for (int i = 0; i < 4; i++) {
        af[i] = frag(&lds[buf][0][(wm * 64 + i * 16 + lo) * 64 + ch]);
        wf[i] = frag(&lds[buf][1][(wn * 64 + i * 16 + lo) * 64 + ch]);
      }
#pragma unroll
      for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < 4; j++) acc[i][j] = mfma16l(wf[i], af[j], acc[i][j]);
    }
    __syncthreads();
  }
  const bool wide = ((a.ldo | a.go) & 3) == 0 && ((size_t)a.out & 7) == 0;
#pragma unroll
  for (int j = 0; j < 4; j++) {
    const int m = m0 + wm * 64 + j * 16 + lo;
    if (m >= rows) continue;
    const int id = list ? list[m] : m;
    const float sc = a.scale ? a.scale[id] : 1.f;
    short* o = (short*)a.out + g * a.go + (long)id * a.ldo;
    if constexpr (GLU) {
#pragma unroll
      for (int i = 0; i < 4; i += 2)
        store_row<true>(a, o, n0 + wn * 32 + i * 8 + 4 * hi, acc[i][j], acc[i + 1][j], sc, wide);
    } else {
#pragma unroll
      for (int i = 0; i < 4; i++)
        store_row<false>(a, o, n0 + wn * 64 + i * 16 + 4 * hi, acc[i][j], acc[i][j], sc, wide);
    }
  }
}

// MF * 16 rows by NF * 16 weight rows (GLU: 16 of gate's and of up's in turn).  The
// waves share the depth: each walks 64 elements at a time of its own part, which
// direct loads bring into a ring of its own in LDS, whole 128-byte lines, without
// barriers, and they add up through LDS.  16 experts of 1536 x 2240, 32 tokens with 4
// each: gate and up 42 us (5.2 TB/s), down 23; 100 tokens 51 and 31.  Fragments
// loaded straight into registers, half a line at a time: 56 and 33, 129 and 65.
template <int MF, int NF, int WAVES, int R, bool GLU>
__global__ __launch_bounds__(WAVES * 64) void grouped_stream_kernel(Grouped a) {
  int g, m0, rows;
  if (!find_rows(a, blockIdx.x, 16 * MF, g, m0, rows)) return;
  constexpr int CHUNK = (MF + NF) * 16 * 64, LOADS = (MF + NF) * 2;
  const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lo = lane & 15, hi = lane >> 4;
  const int n0 = blockIdx.y * (GLU ? NF * 8 : NF * 16);
  __shared__ __attribute__((aligned(16))) short ring[WAVES][R][CHUNK];    // [w rows, a rows]
  g = __builtin_amdgcn_readfirstlane(g);
  const int* list = a.lists ? a.lists + (long)g * a.cap : nullptr;
  const short* A = (const short*)a.a + g * a.ga;
  const short* W = (const short*)a.w + g * a.gw;

  // A load of a wave is 8 rows of 128 bytes, their 16-byte chunks exchanged (xor)
  // by row pair.
  const int chunk = (lane & 7) ^ (lane >> 4);
  const short *wp[NF * 2], *ap[MF * 2];
#pragma unroll
  for (int i = 0; i < NF * 2; i++)
    wp[i] = weight_row<GLU>(a, W, n0, 8 * i + (lane >> 3));
#pragma unroll
  for (int i = 0; i < MF * 2; i++) {
    const int m = min(m0 + 8 * i + (lane >> 3), rows - 1);
    ap[i] = A + (long)((list ? list[m] : m) / a.div) * a.lda;
  }
  const int steps = (a.K + 63) / 64;
  const int first = steps * wid / WAVES, last = steps * (wid + 1) / WAVES;
  auto fetch = [&](int step, int slot) {
    short* at = ring[wid][slot];
    // past the end of a row: its first chunk, not used
    int k[2];
#pragma unroll
    for (int i = 0; i < 2; i++) {
      k[i] = step * 64 + (chunk ^ i << 2) * 8;
      if (k[i] >= a.K) k[i] = 0;
    }
#pragma unroll
    for (int i = 0; i < NF * 2; i++) load_to_lds16(wp[i] + k[i & 1], at + i * 512);
#pragma unroll
    for (int i = 0; i < MF * 2; i++) load_to_lds16(ap[i] + k[i & 1], at + (NF * 2 + i) * 512);
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
      s16x8 v = *reinterpret_cast<const s16x8*>(
          at + (row16 * 16 + lo) * 64 + (((4 * q + hi) ^ (lo >> 1)) << 3));
      if (step * 64 + 32 * q + 8 * hi >= a.K) v = s16x8{};
      return as_frag(v);
    };
    bf16x8l wf[2][NF], af[2][MF];
#pragma unroll
    for (int q = 0; q < 2; q++) {
#pragma unroll
      for (int i = 0; i < NF; i++) wf[q][i] = part(i, q);
#pragma unroll
      for (int j = 0; j < MF; j++) af[q][j] = part(NF + j, q);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");       // read before it is filled again
    if (step + R < last) fetch(step + R, slot);
    slot = slot + 1 == R ? 0 : slot + 1;
#pragma unroll
    for (int q = 0; q < 2; q++)
#pragma unroll
      for (int i = 0; i < NF; i++)
#pragma unroll
        for (int j = 0; j < MF; j++) acc[i][j] = mfma16l(wf[q][i], af[q][j], acc[i][j]);
  }
  __syncthreads();
  // Each wave adds up and stores its share of the tiles, as in linear_rows.hip.  A unit is a
  // tile, or a gate's and its up's.
  constexpr int TILES = GLU ? 2 : 1, UNITS = NF / TILES * MF;
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
  const bool wide = ((a.ldo | a.go) & 3) == 0 && ((size_t)a.out & 7) == 0;
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
    const int m = m0 + 16 * j + lo;
    if (m >= rows) continue;
    const int id = list ? list[m] : m;
    const float sc = a.scale ? a.scale[id] : 1.f;
    short* o = (short*)a.out + g * a.go + (long)id * a.ldo;
    store_row<GLU>(a, o, n0 + (GLU ? i * 8 : i * 16) + 4 * hi, sum[0], sum[TILES - 1], sc, wide);
  }
}

// ---------------------------------------------------------------- routing
// The largest of L neighbouring lanes' values, in all of them: 8, 4, 2 and 1 lanes apart by
// row_ror:8, row_ror:4 and two quad_perm
template <int L>
DEVINL float lanes_max(float v) {
  if constexpr (L == 64) {
    const auto h = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = fmaxf(__uint_as_float(h[0]), __uint_as_float(h[1]));
  }
  if constexpr (L >= 32) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
  }
  v = fmaxf(v, row_move<0x128>(v));
  v = fmaxf(v, row_move<0x124>(v));
  v = fmaxf(v, row_move<0x4e>(v));
  return fmaxf(v, row_move<0xb1>(v));
}

// Top choices of one token's logits z[0..E) in LDS, by L neighbouring lanes; the
// lower index wins a tie.  Not stored unless `store`.  top <= L.  With an expert a lane a
// round is a maximum and a ballot: 16 tokens' 4 of 16 experts 600 cycles, 5000 with the
// lanes' values and indexes exchanged through LDS.
template <int L>
DEVINL void choose(const float* z, int E, int top, int* chosen, float* weight, bool store,
                   int* also = nullptr) {
  const int lane = threadIdx.x & (L - 1);
  float first = 0.f, sum = 0.f, mine = 0.f;
  int pick = 0;
  auto take = [&](int i, float best, int at) {
    if (i == 0) first = best;
    const float p = expf(best - first);
    sum += p;
    if (lane == i) {
      mine = p;
      pick = at;
    }
  };
  if (E <= L) {
    const int group = threadIdx.x & 63 & ~(L - 1);      // its first lane
    float v = lane < E ? z[lane] : -INFINITY;
    v = v == v ? v : -INFINITY;                         // every lane must agree
    bool left = lane < E;
    for (int i = 0; i < top; i++) {
      const float best = lanes_max<L>(left ? v : -INFINITY);
      const unsigned long long all = __ballot(left && v == best) >> group;
      const int at = __ffsll(L == 64 ? all : all & ((1ull << (L & 63)) - 1)) - 1;
      left &= lane != at;
      take(i, best, at);
    }
  } else {
    unsigned long long taken = 0;         // of this lane's experts lane, lane + L, ..
    for (int i = 0; i < top; i++) {
      float best = -INFINITY;
      int at = 1 << 30;
      for (int e = lane, q = 0; e < E; e += L, q++) {
        const float x = z[e] == z[e] ? z[e] : -INFINITY;
        if (!(taken >> q & 1) && (x > best || at == 1 << 30)) {
          best = x;
          at = e;
        }
      }
#pragma unroll
      for (int off = L / 2; off > 0; off >>= 1) {
        const float b = __shfl_xor(best, off);
        const int o = __shfl_xor(at, off);
        if (o != 1 << 30 && (at == 1 << 30 || b > best || (b == best && o < at))) {
          best = b;
          at = o;
        }
      }
      if ((at & (L - 1)) == lane) taken |= 1ull << (at / L);
      take(i, best, at);
    }
  }
  if (store && lane < top) {
    chosen[lane] = pick;
    weight[lane] = mine / sum;
    if (also) also[lane] = pick;
  }
}

template <typename T>
__global__ __launch_bounds__(256) void route_plain_kernel(
    const T* __restrict__ h, const T* __restrict__ wr, const T* __restrict__ bias,
    int* __restrict__ chosen, float* __restrict__ weight, int W, int E, int top) {
  extern __shared__ float z[];
  const long t = blockIdx.x;
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  for (int e = wid; e < E; e += 4) {
    float s = 0.f;
    for (int k = lane; k < W; k += 64) s += ldf(h + t * W + k) * ldf(wr + (long)e * W + k);
    s = wave_sum(s);
    if (lane == 0) z[e] = s + ldf(bias + e);
  }
  __syncthreads();
  if (wid == 0) choose<64>(z, E, top, chosen + t * top, weight + t * top, true);
}

// the rows that chose expert e of n choices, in order, by one wave
DEVINL void list_expert(const int* choices, int n, int e, int* list, int* count) {
  const int lane = threadIdx.x & 63;
  int total = 0;
  for (int base = 0; base < n; base += 64) {
    const bool mine = base + lane < n && choices[base + lane] == e;
    const unsigned long long all = __ballot(mine);
    if (mine) list[total + __popcll(all & ((1ull << lane) - 1))] = base + lane;
    total += __popcll(all);
  }
  if (lane == 0) *count = total;
}

// 16 tokens per workgroup; the waves share the depth.  ET tiles of 16 experts.  A few tokens
// are a chain of loads, so up to 16 experts those of AT steps are asked for at once.  The order
// of the sums is the same for any number of tokens: on it hangs which expert a token at a near
// tie gets, in a short step as in a long prompt.  Experts of 32 tokens of 1536, with this before
// them, 81.1 us with 4 steps as the compiler has them, 77.3 with 4, 77.0 with 12; 16 waves in
// place of four, which add up in another order, 76.6.  4000 tokens and their lists 13.7 us
// with any of these.  With more experts the compiler's 4 steps are 12 to 68 loads by themselves.
// ALL: one workgroup has all tokens, and writes the experts' lists too, for which another
// launch takes 4 us (1, 8 and 16 tokens' experts of 1536 x 2240 29.6 -> 25.9, 58.6 -> 54.6, 68.1
// -> 64.9 us).  Not of more than 16 tokens, whose rows one CU would have to fetch: 32 tokens
// 20500 cycles with the lists, 10300 without them where each 16 have a workgroup.  Nor of
// more than 64 experts, whose lists are too many for four waves: 16 tokens' 8 of 64 of width 1536
// 36.1 -> 19.5 us, but of 128 44.6 -> 50.1, of 256 60.9 -> 74.6.
template <int ET, bool ALL>
__global__ __launch_bounds__(256) void route_mfma_kernel(
    const short* __restrict__ h, const short* __restrict__ wr, const short* __restrict__ bias,
    int* __restrict__ chosen, float* __restrict__ weight, int* __restrict__ lists,
    int* __restrict__ counts, long T, int W, int E, int top) {
  constexpr int AT = ET > 1 ? 1 : 12;
  __shared__ float z[4][16][ET * 16 + 1];
  const long t0 = blockIdx.x * 16L;
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int lo = lane & 15, hi = lane >> 4;
  const short* hp = h + min(t0 + lo, T - 1) * W + 8 * hi;
  f32x4 acc[ET];
#pragma unroll
  for (int i = 0; i < ET; i++) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll(AT == 1 ? 4 : 1)
  for (int k0 = wid * 32; k0 < W; k0 += AT * 128) {
    s16x8 x[AT], y[AT][ET];
#pragma unroll
    for (int a = 0; a < AT; a++) {
      const int k = k0 + 128 * a;
      const bool in = k + 8 * hi < W;
      x[a] = in ? *reinterpret_cast<const s16x8*>(hp + k) : s16x8{};
#pragma unroll
      for (int i = 0; i < ET; i++) {
        const long e = min(16 * i + lo, E - 1);
        y[a][i] = in ? *reinterpret_cast<const s16x8*>(wr + e * W + 8 * hi + k) : s16x8{};
      }
    }
#pragma unroll
    for (int a = 0; a < AT; a++)
      if (k0 + 128 * a < W) {
#pragma unroll
        for (int i = 0; i < ET; i++) acc[i] = mfma16l(as_frag(x[a]), as_frag(y[a][i]), acc[i]);
      }
  }
#pragma unroll
  for (int i = 0; i < ET; i++)
#pragma unroll
    for (int r = 0; r < 4; r++) z[wid][4 * hi + r][16 * i + lo] = acc[i][r];
  __syncthreads();
  for (int i = threadIdx.x; i < 16 * E; i += 256) {
    const int t = i / E, e = i % E;
    z[0][t][e] = z[0][t][e] + z[1][t][e] + z[2][t][e] + z[3][t][e] + bf2f(bias[e]);
  }
  __syncthreads();
  constexpr int L = ET == 1 ? 16 : ET == 2 ? 32 : 64, AT_ONCE = 256 / L;
  __shared__ int picks[ALL ? 16 * ET * 16 : 1];      // [tokens, top]
  for (int t = threadIdx.x / L; t < 16; t += AT_ONCE)
    choose<L>(z[0][t], E, top, chosen + (t0 + t) * top, weight + (t0 + t) * top, t0 + t < T,
              ALL ? picks + t * top : nullptr);
  if constexpr (ALL) {
    __syncthreads();
    for (int e = wid; e < E; e += 4)
      list_expert(picks, (int)T * top, e, lists + (long)e * T, counts + e);
  }
}

// One workgroup per expert: the rows that chose it, in order.  Four choices to a thread at a
// time, for every round waits for its loads and twice at a barrier: 16000 choices of 16
// experts 13.2 us with one each, 5.8 now.
__global__ __launch_bounds__(1024) void expert_lists_kernel(
    const int* __restrict__ chosen, int* __restrict__ lists, int* __restrict__ counts, long n,
    int cap) {
  __shared__ int wave_n[16];
  const int e = blockIdx.x, lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  int* list = lists + (long)e * cap;
  int total = 0;
  for (long base = 0; base < n; base += 4096) {
    const long i = base + 4 * threadIdx.x;
    int c[4];
    if (i + 4 <= n) {
      *reinterpret_cast<int4*>(c) = *reinterpret_cast<const int4*>(chosen + i);
    } else {
#pragma unroll
      for (int j = 0; j < 4; j++) c[j] = i + j < n ? chosen[i + j] : -1;
    }
    int mine = 0;
#pragma unroll
    for (int j = 0; j < 4; j++) mine += c[j] == e;
    int upto = mine;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int x = __shfl_up(upto, off);
      if (lane >= off) upto += x;
    }
    if (lane == 63) wave_n[wid] = upto;
    __syncthreads();
    int at = total + upto - mine;
    for (int w = 0; w < 16; w++) {
      if (w < wid) at += wave_n[w];
      total += wave_n[w];
    }
#pragma unroll
    for (int j = 0; j < 4; j++)
      if (c[j] == e) list[at++] = (int)(i + j);
    __syncthreads();
  }
  if (threadIdx.x == 0) counts[e] = total;
}

// ======================================================== host wrappers ==
// Whether gemm_big.h's kernel pays with `tm` tiles of rows at most: where its tiles of 256
// fill the CUs and their columns.  us, tiles of 128 / it: 16 experts of 1536 x 2240, gate and
// up, 250 rows each (576 tiles) 102 / 82, 1000 rows 299 / 211, down 180 rows (162) 41 / 44, 256
// (192) 68 / 46; 4 experts, 300 rows (144) 33 / 36, 400 (180) 50 / 34; 12 heads of 512 x 128,
// 4000 rows 16.4 / 18.3.  Up to 128 rows half of a tile is empty and it takes a long product:
// 110 rows of 1536 x 2240 65 / 66, 100 of 2048 x 2752 139 / 108, 56 of 3584 x 4096 143 / 95.
// Since what is left after whole rounds is divided, `least` tiles are 96 where all groups have
// as many rows (4 products of 1536 x 1536, 800 rows 30.2 / 29.1, 1300 50 / 37, 600 (72) 24.7 / 28.2;
// of 1024 x 4096, 1500 rows 68.3 / 67.4).  Where they are counted, and fewer than `tm`, 150 down (both
// products, 16 experts of 1536 x 2240, 150 rows 146 / 126), but 176 for gate and up (4 experts of
// 2048 x 2752, 200 rows (154) 77 / 86).
static bool fills_big(long each, long tm, long N, long K, int width, long least) {
  const long tn = (N + width - 1) / width;
  return tm * tn < 1L << 31 && N * 4 >= tn * width * 3 &&
         (each > 128 ? tm * tn >= least : tm * tn * K >= 800000);
}

// ... and takes them: what its 32-bit offsets, whole steps and stores of four columns can do
static bool takes_big(const Grouped& a, long each, long tm, int width) {
  return a.G <= 64 && a.K > 0 && a.K % 64 == 0 && a.N % 4 == 0 && (a.ldo | a.go) % 4 == 0 &&
         (uintptr_t)a.out % 8 == 0 && a.K < 1L << 22 && a.ldw < 1L << 22 &&
         (a.rows / a.div + 1) * a.lda < 1L << 31 &&
         fills_big(each, tm, a.N, a.K, width, !a.lists ? 96 : width < BIG ? 176 : 150);
}

// Whether T rows of each of G products fill gemm_big.h's tiles, for those that are the library's
// else
bool group_linear_fills(long T, long G, long N, long K) {
  return fills_big(T, G * ((T + BIG - 1) / BIG), N, K, BIG, 176);
}

template <bool GLU>
static void launch_grouped(const Grouped& a, bool bf16) {
  if (a.rows == 0 || a.N == 0) return;
  auto stream = at::hip::getCurrentHIPStream();
  // row-tiles that any distribution of the rows over the groups may need
  auto tiles_of = [&](long bm) {
    return a.lists ? std::min<long>(a.rows / bm + a.G, a.rows) : a.G * ((a.rows + bm - 1) / bm);
  };
  const bool mfma = bf16 && a.K % 8 == 0 && (a.lda | a.ga | a.ldw | a.gw | a.up) % 8 == 0 &&
                    (uintptr_t)a.a % 16 == 0 && (uintptr_t)a.w % 16 == 0;
  if (mfma) {
    const long each = a.lists ? a.rows / a.G : a.rows;      // rows of a group, about
    const long tm = tiles_of(128), tn = (a.N + (GLU ? 63 : 127)) / (GLU ? 64 : 128);
    // Up to 52 rows the weights are what counts: 160 tokens with 4 of 16 experts of 1536 x
    // 2240 68 and 34 us in rows of 64, 79 and 39 in tiles; 288 tokens 84 and 51 against 80
    // and 44.  Unless there are more than 32 rows to each and tiles enough for rounds of
    // their own, the more the longer a tile takes: 40 rows of 128 experts of 512 x 1024 (1024
    // tiles) 49 us against 58, of 16 experts of 4096 x 3584 (900) 253 against 207.
    const bool many = tm * tn >= std::max<long>(256, a.K / 2);
    const long big = tiles_of(BIG);
    if (each > 52 && takes_big(a, each, big, GLU ? BIG / 2 : BIG)) {
      Big p{};
      p.x = (const short*)a.a;
      p.w = (const short*)a.w;
      p.w2 = p.w + a.up;
      p.y = (short*)a.out;
      p.ldy = a.ldo;
      p.M = a.rows;
      p.N = a.N;
      p.K = a.K;
      p.lists = a.lists;
      p.counts = a.lists ? a.counts : nullptr;
      p.scale = a.scale;
      p.cap = a.cap;
      p.div = a.div;
      p.G = a.G;
      p.ldx = a.lda;
      p.ldw = a.ldw;
      p.gx = a.ga;
      p.gw = a.gw;
      p.gy = a.go;
      launch_big_grouped<GLU ? SILU_GLU : NO_ACT>(p, big);
      HIP_CHECK_LAST();
      return;
    }
    if (each > 52 ? each > 512 || tm * tn >= 64 : each > 32 && many) {
      TORCH_CHECK(tm * tn < (1L << 31));
      hipLaunchKernelGGL((grouped_tiles_kernel<GLU>), dim3(tm * tn), dim3(256), 0, stream, a,
                         (int)tm, (int)tn);
    } else {
      // 64 rows at a time read the weights once but leave half the workgroups: where there
      // are enough for every CU all the same, and the depth is worth it.  8 experts of 1024 x
      // 512, 40 rows each: 13 and 10 us with 32 rows, 18 and 14 with 64.  More than 52
      // rows come here in small grids only: 12 heads of 512 x 128, 128 rows 6.2 us with 32, 7.6
      // with 64.
      constexpr long WIDE = GLU ? 32 : 64;
      const bool full =
          a.lists ? std::min<long>(tiles_of(64), a.rows) * ((a.N + WIDE - 1) / WIDE) >= 256
                  : tiles_of(32) * ((a.N + WIDE / 2 - 1) / (WIDE / 2)) > 256;
      const int mf = each > 28 && each <= 52 && a.K >= 1024 && !many && full ? 4
                     : each > 12 ? 2 : 1;
      // Four waves with a chunk of their own each.  Where 64 weight rows to a workgroup
      // leave CUs idle, 32 and two chunks: one token's 4 experts of 1536 x 2240 7.7 us
      // against 10; and for a few rows' gate and up of some depth: 16 experts of 1536 x 2240
      // 42.4 us, 43.9 with 64 rows, of 4096 x 3584 138 and 143, down 24.5 and 22.9.  Both products,
      // 12 rows each: 64 experts of 512 x 1408 72 and 62, 32 of 1024 x 1024 44.0 and 43.8, 64 of
      // 1536 x 512 58.1 and 59.5, 16 of 4096 x 3584 279 and 291.
      const long busy = std::min<long>(tiles_of(16 * mf), a.rows);
#define STREAM(MF, NF, R)                                                                      \
  hipLaunchKernelGGL((grouped_stream_kernel<MF, NF, 4, R, GLU>),                               \
                     dim3(tiles_of(16 * MF), (a.N + NF * (GLU ? 8 : 16) - 1) /                 \
                                                 (NF * (GLU ? 8 : 16))),                       \
                     dim3(256), 0, stream, a)
      if (busy * ((a.N + (GLU ? 31 : 63)) / (GLU ? 32 : 64)) < 256) {
        if (mf == 4) STREAM(4, 2, 2);
        else if (mf == 2) STREAM(2, 2, 2);
        else STREAM(1, 2, 2);
      } else if (mf == 4) {
        STREAM(4, 4, 1);
      } else if (mf == 2) {
        STREAM(2, 4, 1);
      } else if (GLU && a.K >= 1536) {
        STREAM(1, 2, 2);
      } else {
        STREAM(1, 4, 1);
      }
#undef STREAM
    }
    HIP_CHECK_LAST();
    return;
  }
  const long tiles = tiles_of(64);
  const dim3 grid((a.N + 63) / 64, tiles);
  TORCH_CHECK(tiles <= 65535, "batch too large for the plain grouped product");
  if (bf16)
    hipLaunchKernelGGL((grouped_plain_kernel<short, GLU>), grid, dim3(256), 0, stream, a);
  else
    hipLaunchKernelGGL((grouped_plain_kernel<float, GLU>), grid, dim3(256), 0, stream, a);
  HIP_CHECK_LAST();
}

static bool is_bf16(const torch::Tensor& t) {
  TORCH_CHECK(t.is_cuda());
  if (t.scalar_type() == torch::kBFloat16) return true;
  TORCH_CHECK(t.scalar_type() == torch::kFloat32, "bf16 or float32 expected");
  return false;
}

void group_linear(torch::Tensor x, torch::Tensor w, torch::Tensor out) {
  on_gpu({x, w, out});
  const long T = x.size(0), G = x.size(1), K = x.size(2), N = w.size(1);
  TORCH_CHECK(x.dim() == 3 && w.dim() == 3 && out.dim() == 3 && w.size(0) == G && w.size(2) == K &&
              out.size(0) == T && out.size(1) == G && out.size(2) == N);
  TORCH_CHECK(x.stride(2) == 1 && w.stride(2) == 1 && out.stride(2) == 1);
  TORCH_CHECK(w.scalar_type() == x.scalar_type() && out.scalar_type() == x.scalar_type());
  Grouped a{};
  a.a = x.data_ptr();
  a.w = w.data_ptr();
  a.out = out.data_ptr();
  a.lda = x.stride(0);
  a.ga = x.stride(1);
  a.ldw = w.stride(1);
  a.gw = w.stride(0);
  a.ldo = out.stride(0);
  a.go = out.stride(1);
  a.rows = T;
  a.div = 1;
  a.G = G;
  a.N = N;
  a.K = K;
  launch_grouped<false>(a, is_bf16(x));
}

std::vector<torch::Tensor> moe_route(torch::Tensor h, torch::Tensor router, torch::Tensor bias,
                                     long top) {
  on_gpu({h, router, bias});
  TORCH_CHECK(h.dim() == 2 && h.is_contiguous() && router.is_contiguous() && bias.is_contiguous());
  const long T = h.size(0), W = h.size(1), E = router.size(0);
  TORCH_CHECK(router.size(1) == W && bias.numel() == E && router.scalar_type() == h.scalar_type() &&
              bias.scalar_type() == h.scalar_type());
  TORCH_CHECK(top >= 1 && top <= E && top <= 64 && E <= 4096, "unsupported number of experts");
  auto ints = h.options().dtype(torch::kInt);
  auto chosen = torch::empty({T, top}, ints);
  auto weight = torch::empty({T, top}, h.options().dtype(torch::kFloat32));
  auto lists = torch::empty({E, T}, ints);
  auto counts = torch::empty({E}, ints);
  TORCH_CHECK(T > 0 && T * top < (1L << 31));
  auto stream = at::hip::getCurrentHIPStream();
#define ROUTE_OF(ET, ALL)                                                                      \
  hipLaunchKernelGGL((route_mfma_kernel<ET, ALL>), dim3((T + 15) / 16), dim3(256), 0, stream,  \
                     (const short*)h.data_ptr(), (const short*)router.data_ptr(),              \
                     (const short*)bias.data_ptr(), chosen.data_ptr<int>(),                    \
                     weight.data_ptr<float>(), lists.data_ptr<int>(), counts.data_ptr<int>(),  \
                     T, (int)W, (int)E, (int)top)
#define ROUTE(ET)                              \
  do {                                         \
    listed = T <= 16 && ET <= 4;               \
    if (listed) ROUTE_OF(ET, (ET <= 4));       \
    else ROUTE_OF(ET, false);                  \
  } while (0)
  bool listed = false;
  if (is_bf16(h) && W % 8 == 0 && E <= 256 && (uintptr_t)h.data_ptr() % 16 == 0 &&
      (uintptr_t)router.data_ptr() % 16 == 0) {
    if (E <= 16) ROUTE(1);
    else if (E <= 32) ROUTE(2);
    else if (E <= 64) ROUTE(4);
    else if (E <= 128) ROUTE(8);
    else ROUTE(16);
  } else if (is_bf16(h))
    hipLaunchKernelGGL((route_plain_kernel<short>), dim3(T), dim3(256), 4 * E, stream,
                       (const short*)h.data_ptr(), (const short*)router.data_ptr(),
                       (const short*)bias.data_ptr(), chosen.data_ptr<int>(),
                       weight.data_ptr<float>(), (int)W, (int)E, (int)top);
  else
    hipLaunchKernelGGL((route_plain_kernel<float>), dim3(T), dim3(256), 4 * E, stream,
                       (const float*)h.data_ptr(), (const float*)router.data_ptr(),
                       (const float*)bias.data_ptr(), chosen.data_ptr<int>(),
                       weight.data_ptr<float>(), (int)W, (int)E, (int)top);
#undef ROUTE
#undef ROUTE_OF
  if (!listed)
    hipLaunchKernelGGL(expert_lists_kernel, dim3(E), dim3(1024), 0, stream,
                       chosen.data_ptr<int>(), lists.data_ptr<int>(), counts.data_ptr<int>(),
                       T * top, (int)T);
  HIP_CHECK_LAST();
  return {chosen, weight, lists, counts};
}

static void check_lists(const torch::Tensor& lists, const torch::Tensor& counts, long E) {
  on_gpu({lists, counts});
  TORCH_CHECK(lists.scalar_type() == torch::kInt && lists.is_contiguous() &&
              lists.dim() == 2 && lists.size(0) == E);
  TORCH_CHECK(counts.scalar_type() == torch::kInt && counts.is_contiguous() && counts.numel() == E);
}

// [T * top, ff]: silu(gate h) * (up h) of every choice
torch::Tensor moe_gate_up(torch::Tensor h, torch::Tensor gate_up, torch::Tensor lists,
                          torch::Tensor counts, long top) {
  const long T = h.size(0), W = h.size(1), E = gate_up.size(0), ff = gate_up.size(2);
  on_gpu({h, gate_up});
  TORCH_CHECK(h.dim() == 2 && h.is_contiguous() && gate_up.dim() == 4 && gate_up.is_contiguous() &&
              gate_up.size(1) == 2 && gate_up.size(3) == W &&
              gate_up.scalar_type() == h.scalar_type());
  check_lists(lists, counts, E);
  TORCH_CHECK(lists.size(1) == T);
  auto act = torch::empty({T * top, ff}, h.options());
  Grouped a{};
  a.a = h.data_ptr();
  a.w = gate_up.data_ptr();
  a.out = act.data_ptr();
  a.lda = W;
  a.ldw = W;
  a.up = ff * W;
  a.gw = 2 * ff * W;
  a.ldo = ff;
  a.lists = lists.data_ptr<int>();
  a.counts = counts.data_ptr<int>();
  a.rows = T * top;
  a.cap = T;
  a.div = top;
  a.G = E;
  a.N = ff;
  a.K = W;
  launch_grouped<true>(a, is_bf16(h));
  return act;
}

// [T, top, W]: down act, times the choice's weight
torch::Tensor moe_down(torch::Tensor act, torch::Tensor down, torch::Tensor lists,
                       torch::Tensor counts, torch::Tensor weights) {
  const long T = weights.size(0), top = weights.size(1), E = down.size(0), W = down.size(1),
             ff = down.size(2);
  on_gpu({act, down, weights});
  TORCH_CHECK(act.dim() == 2 && act.is_contiguous() && down.dim() == 3 && down.is_contiguous() &&
              act.size(0) == T * top && act.size(1) == ff && act.scalar_type() == down.scalar_type());
  TORCH_CHECK(weights.scalar_type() == torch::kFloat32 && weights.is_contiguous());
  check_lists(lists, counts, E);
  TORCH_CHECK(lists.size(1) == T);
  auto y = torch::empty({T, top, W}, act.options());
  Grouped a{};
  a.a = act.data_ptr();
  a.w = down.data_ptr();
  a.out = y.data_ptr();
  a.lda = ff;
  a.ldw = ff;
  a.gw = W * ff;
  a.ldo = W;
  a.lists = lists.data_ptr<int>();
  a.counts = counts.data_ptr<int>();
  a.scale = weights.data_ptr<float>();
  a.rows = T * top;
  a.cap = T;
  a.div = 1;
  a.G = E;
  a.N = W;
  a.K = ff;
  launch_grouped<false>(a, is_bf16(act));
  return y;
}
