// bf16 products of many rows, y = x w^T, in tiles of 256 x 256: with an adapter's
// rank-64 pair as one more step of the depth and a bias (lora.hip), or of a gated
// feed-forward's two weights at once, whose columns meet before they are rounded
// (glu.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <ATen/hip/HIPContext.h>

#include <type_traits>

#include "common.h"

typedef __bf16 bf16x8_m __attribute__((ext_vector_type(8)));

constexpr int BIG = 256;

// ACT: a tile has 128 columns of y; of every 64 rows of its w tile the first half is
// w's and the second the same columns of w2, and y = act(x w) * (x w2).
// SILU_KEEP: silu of both products rounded, which are stored too, side by side in `kept` [M, 2 N]
// (what a backward wants of them); the adapter's pair for both.
// ROPE: y's 256 columns are heads of q, k and v, whose halves (of 32 or 64) take the places of w's
// and w2's columns; they are rounded, turned by the row's position, and go to q, k and v.
enum { NO_ACT, SILU_GLU, GELU_GLU, SILU_KEEP, ROPE };
constexpr int big_columns(int act) { return act == NO_ACT || act == ROPE ? BIG : BIG / 2; }
enum { NO_BIAS, BIAS_F32, BIAS_BF16 };    // bf16: of an even N, on 4 bytes

template <int ACT>
DEVINL float glu(float g, float up) {
  // swiglu_fwd_kernel's steps, bit by bit: the exact quotient, which its backward has too
  if (ACT == SILU_KEEP) return g * (1.f / (1.f + __expf(-g))) * up;
  const float z = ACT == SILU_GLU ? g : 1.5957691216057308f * (g + 0.044715f * g * g * g);
  return g * __builtin_amdgcn_rcpf(1.f + __expf(-z)) * up;      // gelu_tanh: x sigmoid(2 ..)
}

// Into how many units of fewer rows the tiles are divided that are left after whole rounds of
// the CUs: where they still fit one round.
__host__ __device__ inline int parts_of(int left, int cus) {
  return left == 0 || left * 2 > cus ? 1 : left * 4 > cus ? 2 : 4;
}

struct Big {
  const short *x, *w;            // [M, K], [N, K]
  const short *u, *b;            // [M, 64], [N, 64]
  const void* bias;              // [N], as BIAS says
  const short* w2;               // as w
  short* y;
  long ldy;
  short* kept;
  short *q, *k, *v;              // [M, Hq, 2 half], [M, Hkv, 2 half]
  const float* table;            // cos | sin [positions, 2 half]
  const long* pos;               // [M]
  int half, Hq, Hkv;
  int M, N, K, grid_m, grid_n;
  int whole, parts, units;       // tiles that are one unit of work, and units of the others
  int cus;                       // grouped: what these are divided for
  // grouped: G <= 64 products, of the rows that lists [G, cap] name (of x a row / div) or of
  // M each; their results go to the same rows of y, times scale [rows]
  const int *lists, *counts;
  const float* scale;
  int cap, div, G;
  long ldx, ldw, gx, gw, gy;     // row and group strides
};

DEVINL void load_big(const void* base, unsigned offset, unsigned at) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
               ::"s"(at), "v"(offset), "s"(in_sgprs(base)) : "memory");
}

// One workgroup of 8 waves per CU walks over tiles; a wave has 128 rows and 64 columns
// (or both weights' 32).  The two halves of the workgroup are half a phase apart: on every
// SIMD one wave's 16 products run while the other one reads LDS and asks for memory,
// and then they change places at a barrier.  A phase is a quarter of the wave's tile
// and one step of 64 of the depth: x's rows and w's columns in halves, of which one
// changes from phase to phase; what a phase multiplies was read a phase earlier.  LDS has
// two steps, in quarters of 16 KB that are asked for again as soon as their last reader is
// two phases away, so that a load has a whole step's time.
//
// Products are 16x16x32: by themselves they reach 1.88 PFLOP/s on normally distributed
// data, 32x32x16 1.64 (the part lowers its clock, to 1.9 GHz where zeros keep 2.4, and those
// move twice as much of the sums).  x is the first operand and w's rows are dealt to LDS so that a lane
// ends up with 4 neighbouring columns of y and 16 lanes with 128 bytes: stores of 16 bytes
// to 64 rows' quarter lines cost up to 10%.  They are marked as not to be kept, which makes
// no difference, neither to a large y nor to a small one that the next kernel reads at once:
// with SwiGLU behind it 212 x 1152 x 896 19.8 us and 19.7 without the mark, 500 x 17920 x 1536
// 41.8 and 41.9, 46673 x 17920 x 1536 2529 and 2521.  The next tile's first two steps are asked
// for before the stores.
//
// 8192 x 8192 x 8192: 0.71 ms (1530 TFLOP/s), 48720 x 17920 x 1536 + 64: 2.13 (1310),
// 48720 x 1536 x 8960 + 64: 1.01 (1340).  Lockstep waves that all read, then all
// multiply 32x32x16, a barrier a step: 0.88 (1250), 2.70 (1030), 1.21 (1120).
template <bool HAS_LORA, int BIAS, bool VEC, int ACT, bool GROUPED = false>
__global__ __launch_bounds__(512, 2) void gemm_big_kernel(Big p) {
  constexpr int TN = big_columns(ACT);
  constexpr int STORES = ACT == SILU_KEEP ? 48 : TN / 8;               // of a wave and whole tile
  static_assert((ACT != SILU_KEEP && ACT != ROPE) || (VEC && !GROUPED));
  static_assert(ACT != ROPE || (!HAS_LORA && BIAS != BIAS_F32));
  constexpr int STEP = BIG * 128;                                      // bytes
  __shared__ __attribute__((aligned(16))) short lds[2][2][BIG * 64];   // x's two steps, w's
  __shared__ float biases[2][BIAS ? 2 * BIG : 1];
  // of groups: tiles of rows before each, and its rows; of a unit's rows: where they go
  __shared__ int starts[GROUPED ? 65 : 1], sizes[GROUPED ? 64 : 1], ids[2][GROUPED ? BIG : 1];
  __shared__ float scales[2][GROUPED ? BIG : 1];
  __shared__ int turns[2][ACT == ROPE ? BIG : 1];         // the tile's rows' positions
  const int tid = threadIdx.x, lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wn = (wid & 3) * 64;
  const int n_k1 = p.K >> 6, n_kt = n_k1 + (HAS_LORA ? 1 : 0);

  int grid_m = p.grid_m, units = p.units, whole = p.whole, left_parts = p.parts, M = p.M, g = 0;
  if constexpr (GROUPED) {
    if (wid == 0) {
      const int c = lane >= p.G ? 0 : p.counts ? p.counts[lane] : p.M;
      int s = (c + BIG - 1) / BIG;
#pragma unroll
      for (int off = 1; off < 64; off <<= 1) {
        const int y = __shfl_up(s, off);
        if (lane >= off) s += y;
      }
      sizes[lane] = c;
      starts[lane + 1] = s;
      if (lane == 0) starts[0] = 0;
    }
    __syncthreads();
    grid_m = __builtin_amdgcn_readfirstlane(starts[64]);
    const int tiles = grid_m * p.grid_n, left = tiles % p.cus;
    left_parts = parts_of(left, p.cus);
    whole = left_parts > 1 ? tiles - left : tiles;
    units = whole + (tiles - whole) * left_parts;
    if (blockIdx.x >= units) return;
  }

  // unit `at`: the tile's place, and which rows of it
  int m0, n0, parts;
  auto place = [&](int at) {
    int wg = at, part = 0;
    parts = 1;
    if (at >= whole) {
      parts = left_parts;
      wg = whole + (at - whole) / parts;
      part = (at - whole) % parts;
    }
    const int nwg = grid_m * p.grid_n, q = nwg >> 3, r = nwg & 7;
    const int xcd = wg & 7, i = wg >> 3;
    wg = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + i;
    constexpr int GM = 8;       // tiles that run together share rows and columns
    const int group = wg / (GM * p.grid_n), first = group * GM;
    const int rows_here = min(GM, grid_m - first);
    const int tile = first + (wg - group * GM * p.grid_n) % rows_here;
    m0 = tile * BIG + part * (BIG / parts);
    n0 = (wg - group * GM * p.grid_n) / rows_here * TN;
    if constexpr (GROUPED) {
      const int l = threadIdx.x & 63;
      g = __ffsll((unsigned long long)__ballot(tile >= starts[l] && tile < starts[l + 1])) - 1;
      m0 = (tile - __builtin_amdgcn_readfirstlane(starts[g])) * BIG + part * (BIG / parts);
      M = __builtin_amdgcn_readfirstlane(sizes[g]);
      // a group's last rows: of a tile's parts the first has all of them
      if (parts == 1 && M - m0 <= BIG / 2) parts = M - m0 <= BIG / 4 ? 4 : 2;
    }
  };

  // what follows from the lane, made again where it is needed: kept over the loop it
  // would cost the loop's registers
  auto fresh_tid = [&] {
    int t = tid;
    asm volatile("" : "+v"(t));
    return t;
  };
  // A quarter is 128 rows of LDS: of x rows 0-63 and 128-191 (or 64 on), of w rows 0-31,
  // 64-95, .. (or 32 on); a thread has one 16-byte chunk of two of them.  Chunks are
  // exchanged (xor) by row pair, for two rows fill the banks.  Of a part of a tile only
  // x's first half is there, 128 / parts rows for each half of the workgroup.
  unsigned xo[4], wo[4];
  int side = 0;
  auto x_offsets = [&](int ld) {
    const int t = fresh_tid(), r = t >> 3, c = ((t & 7) ^ (r >> 1 & 7)) << 3;
#pragma unroll
    for (int h = 0; h < 4; h++) {
      const int m = parts == 1 ? r + 64 * (h >> 1) + 128 * (h & 1)
                               : min(r, 128 / parts - 1) + 128 / parts * (h & 1);
      if constexpr (GROUPED) {
        const int row = min(m0 + m, M - 1);
        const int id = p.lists ? p.lists[(long)g * p.cap + row] : row;
        if ((t & 7) == 0) {
          ids[side][m] = id;
          scales[side][m] = p.scale ? p.scale[id] : 1.f;
        }
        xo[h] = ((unsigned)(p.div > 1 ? id / p.div : id) * (unsigned)ld + c) * 2;
      } else {
        xo[h] = (unsigned)(min(m, max(M - 1 - m0, 0)) * ld + c) * 2;
      }
    }
  };
  // first column of the halves that 64 rows of LDS hold, the i-th of four
  auto first_half = [&](int i) { return p.half == 32 ? 64 * i : (i >> 1) * 128 + (i & 1) * 32; };
  // LDS row 16 t + l of 64 is column 4 l + t, or 2 l + t % 2 of w (t < 2) or w2
  auto w_offsets = [&](int ld) {
    const int t = fresh_tid(), r = t >> 3 & 31, l = r & 15;
    const int c = ((t & 7) ^ (r >> 1 & 7)) << 3;
    if constexpr (ACT == ROPE) {
#pragma unroll
      for (int h = 0; h < 4; h++)
        wo[h] = (unsigned)(min(2 * l + (r >> 4) + first_half((t >> 8) + 2 * (h & 1)),
                               p.N - 1 - p.half - n0) * ld + c) * 2;
      return;
    }
#pragma unroll
    for (int h = 0; h < 4; h++) {
      const int n = ACT ? 2 * l + (r >> 4) + (t >> 8) * 32 + 64 * (h & 1)
                        : 4 * l + (r >> 4) + 2 * (h >> 1) + (t >> 8) * 64 + 128 * (h & 1);
      wo[h] = (unsigned)(min(n, p.N - 1 - n0) * ld + c) * 2;
    }
  };
  const short *xb, *wb, *w2b, *ub, *bb, *b2b;
  const unsigned base =
      (unsigned)(size_t)(const __attribute__((address_space(3))) short*)&lds[0][0][0];
  const unsigned xat = base + wid * 1024, wat = base + 2 * STEP + ((wid & 3) * 8 + (wid >> 2) * 64) * 128;
  auto load_x = [&](int kt, int h) {
    if (HAS_LORA && kt == n_k1 && h == 0) x_offsets(64);
    const short* src = HAS_LORA && kt == n_k1 ? ub : xb + kt * 64;
#pragma unroll
    for (int i = 0; i < 2; i++)
      load_big(src, xo[2 * h + i], xat + (kt & 1) * STEP + (64 * h + 128 * i) * 128);
  };
  auto load_w = [&](int kt, int h, bool first) {
    if (HAS_LORA && kt == n_k1 && first) w_offsets(64);
    const short* src = HAS_LORA && kt == n_k1 ? (h ? b2b : bb) : (h ? w2b : wb) + kt * 64;
#pragma unroll
    for (int i = 0; i < 2; i++)
      load_big(src, wo[2 * h + i], wat + (kt & 1) * STEP + (32 * h + 128 * i) * 128);
  };
  auto begin = [&] {            // the first two steps of the unit at m0, n0
    x_offsets(GROUPED ? p.ldx : p.K);
    w_offsets(GROUPED ? p.ldw : p.K);
    const int row = min(m0, M - 1);       // a part of the last tile may have none
    xb = GROUPED ? p.x + g * p.gx : p.x + (long)row * p.K;
    const long first_w = GROUPED ? g * p.gw + n0 * p.ldw : (long)n0 * p.K;
    wb = p.w + first_w;
    w2b = ACT == ROPE ? wb + (long)p.half * p.K : ACT ? p.w2 + first_w : wb;
    if (HAS_LORA) {
      ub = p.u + (long)row * 64;
      bb = p.b + (long)n0 * 64;
      b2b = ACT ? bb + (long)p.N * 64 : bb;
    }
    if (BIAS == BIAS_F32)
      load_to_lds4(p.bias, (unsigned)min(n0 + wn + lane, p.N - 1) * 4, &biases[side][wid * 64]);
    if (BIAS == BIAS_BF16) {      // two columns a lane
      const int n = ACT == ROPE ? first_half(wid & 3) + (lane & 15) * 2 + (lane >> 4 & 1) * p.half
                                : wn + 2 * lane;
      load_to_lds4(p.bias, (unsigned)min(n0 + n, p.N - 2) * 2, &biases[side][wid * 64]);
    }
    if (ACT == ROPE) {            // their low words
      const int r = (wid & 3) * 64;
      load_to_lds4(p.pos, (unsigned)min(m0 + r + lane, p.M - 1) * 8, &turns[side][r]);
    }
    load_x(0, 0);
    load_w(0, 0, true);
    load_w(0, 1, false);
    load_x(0, 1);
    if (n_kt > 1) {
      load_x(1, 0);
      load_w(1, 1, true);
      load_w(1, 0, false);
      load_x(1, 1);
    }
  };

  unsigned xa[2], wa[2];        // of each 32 of a step's depth
#pragma unroll
  for (int ks = 0; ks < 2; ks++) {
    const int lo = lane & 15, hi = lane >> 4, xr = (wid >> 2) * 128 + lo, wr = wn + lo;
    xa[ks] = base + xr * 128 + (((4 * ks + hi) ^ (xr >> 1 & 7)) << 4);
    wa[ks] = base + 2 * STEP + wr * 128 + (((4 * ks + hi) ^ (wr >> 1 & 7)) << 4);
  }
  auto lds_frag = [](unsigned at) {
    typedef __attribute__((address_space(3))) const char* lds_bytes;
    typedef __attribute__((address_space(3))) const bf16x8_m* lds_m;
    return *(lds_m)((lds_bytes)0 + at);
  };
  bf16x8_m xf[2][2][4], wf[2][2][2];       // [half][32 of the depth][tile]
  f32x4 acc[8][2][2];                      // [tile of rows][half of the columns][tile]
  auto read_x = [&](int buf, int h, int ks, int t) {
    xf[h][ks][t] = lds_frag(xa[ks] + buf * STEP + (4 * h + t) * 2048);
  };
  auto read_w = [&](int buf, int h) {
#pragma unroll
    for (int e = 0; e < 4; e++)
      wf[h][e >> 1][e & 1] = lds_frag(wa[e >> 1] + buf * STEP + h * 4096 + (e & 1) * 2048);
  };
  auto barrier = [&] {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
  auto products = [&](int h, int j) {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int t2 = 0; t2 < 4; t2 += 2) {
      if ((4 * h + t2) * parts >= 8) continue;
#pragma unroll
      for (int ks = 0; ks < 2; ks++)
#pragma unroll
        for (int t = t2; t < t2 + 2; t++)
#pragma unroll
          for (int e = 0; e < 2; e++)
            acc[4 * h + t][j][e] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                xf[h][ks][t], wf[j][ks][e], acc[4 * h + t][j][e], 0, 0, 0);
    }
    __builtin_amdgcn_s_setprio(0);
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    barrier();
  };
  // Step kt of the depth.  F: which of w's halves comes first (the one that the step
  // before had last), FIRST: the last tile's stores may be under way.  The waits are
  // for the quarter that is read next, and leave the younger ones' loads (and stores) be.
  auto step = [&](auto f, auto is_first, int kt) {
    constexpr int F = decltype(f)::value, S = 1 - F;
    constexpr bool FIRST = decltype(is_first)::value;
    constexpr int E = FIRST ? STORES : 0;
    const bool more = kt + 2 < n_kt, next = kt + 1 < n_kt;
    read_w(F, S);
    read_x(F, 1, 0, 0);
    read_x(F, 1, 0, 1);
    if (!FIRST && next) load_x(kt + 1, 1);
    barrier();
    products(0, F);

    read_x(F, 1, 0, 2);
    read_x(F, 1, 0, 3);
#pragma unroll
    for (int t = 0; t < 4; t++) read_x(F, 1, 1, t);
    if (more) {
      load_x(kt + 2, 0);
      wait_loads<8 + E>();
    } else {
      wait_loads<6 + E>();
    }
    barrier();
    products(0, S);

#pragma unroll
    for (int t = 0; t < 4; t++) read_x(S, 0, 0, t);
    read_x(S, 0, 1, 0);
    read_x(S, 0, 1, 1);
    if (more) {
      load_w(kt + 2, F, true);
      wait_loads<8 + E>();
    } else {
      wait_loads<4 + E>();
    }
    barrier();
    products(1, S);

    read_x(S, 0, 1, 2);
    read_x(S, 0, 1, 3);
    read_w(S, S);
    if (more) {
      load_w(kt + 2, S, false);
      wait_loads<6 + E>();
    } else {
      wait_loads<E>();
    }
    barrier();
    products(1, F);
  };
  typedef std::integral_constant<int, 0> Zero;
  typedef std::integral_constant<int, 1> One;

  place(blockIdx.x);
  begin();
  wait_loads<0>();
  for (int at = blockIdx.x;;) {
    if (n_kt > 1) wait_loads<8 + STORES>();
    else wait_loads<STORES>();
    barrier();
#pragma unroll
    for (int i = 0; i < 8; i++)
#pragma unroll
      for (int j = 0; j < 4; j++) acc[i][j >> 1][j & 1] = f32x4{};
#pragma unroll
    for (int t = 0; t < 8; t++) read_x(0, 0, t >> 2, t & 3);
    read_w(0, 0);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if (wid >= 4) barrier();
    step(Zero(), std::true_type(), 0);
    for (int kt = 1; kt < n_kt; kt += 2) {
      step(One(), std::false_type(), kt);
      if (kt + 1 < n_kt) step(Zero(), std::false_type(), kt + 1);
    }
    if (wid < 4) barrier();

    const int m1 = m0, n1 = n0, parts1 = parts, side1 = side, M1 = M;
    short* const y1 = GROUPED ? p.y + g * p.gy : p.y;
    at += gridDim.x;
    const bool another = at < units;
    if (another) {
      place(at);
      side ^= 1;
      begin();
    }
    // lane: row 16 i + 4 hi + r of its half's, columns 4 (2) lo + 0 .. of the wave's
    const int t = fresh_tid() & 63, lo = t & 15, hi = t >> 4;
    const int gm0 = m1 + (wid >> 2) * (128 / parts1) + 4 * hi;
    // row gm of y, and what it is multiplied by
    auto row_of = [&](int gm) { return y1 + (GROUPED ? ids[side1][gm - m1] : gm) * p.ldy; };
    auto scale_of = [&](int gm) { return GROUPED ? scales[side1][gm - m1] : 1.f; };
    if constexpr (ACT == NO_ACT) {
      const int gn = n1 + wn + 4 * lo;
      float bv[4];
      if (BIAS) {
#pragma unroll
        for (int c = 0; c < 4; c++)
          bv[c] = BIAS == BIAS_F32
                      ? biases[side1][wid * 64 + 4 * lo + c]
                      : bf2f(reinterpret_cast<const short*>(&biases[side1][wid * 64])[4 * lo + c]);
      }
#pragma unroll
      for (int i = 0; i < 8; i++) {
        if (i * parts1 >= 8) continue;
#pragma unroll
        for (int r = 0; r < 4; r++) {
          const int gm = gm0 + 16 * i + r;
          float v[4];
#pragma unroll
          for (int c = 0; c < 4; c++) v[c] = acc[i][c >> 1][c & 1][r] + (BIAS ? bv[c] : 0.f);
          if (gm >= M1) continue;
          short* dst = row_of(gm) + gn;
          if (GROUPED) {
            const float sc = scale_of(gm);
#pragma unroll
            for (int c = 0; c < 4; c++) v[c] *= sc;
          }
          if (VEC) {
            typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
            if (gn < p.N)
              __builtin_nontemporal_store(u32x2{pack2bf(v[0], v[1]), pack2bf(v[2], v[3])},
                                          reinterpret_cast<u32x2*>(dst));
          } else {
#pragma unroll
            for (int c = 0; c < 4; c++)
              if (gn + c < p.N) dst[c] = f2bf(v[c]);
          }
        }
      }
    } else if constexpr (ACT == ROPE) {
      typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
      typedef float f32x2 __attribute__((ext_vector_type(2)));
      const int D = 2 * p.half, n = n1 + first_half(wid & 3), d = n % D, head = n / D;
      const bool is_q = head < p.Hq, is_v = head >= p.Hq + p.Hkv;
      const long ld = (long)(is_q ? p.Hq : p.Hkv) * D;
      short* const to = (is_q ? p.q + head * D : is_v ? p.v + (head - p.Hq - p.Hkv) * D
                                                      : p.k + (head - p.Hq) * D) + d;
      const bool odd = lo & 1, in = n < p.N;
      f32x2 bv[2] = {};
      if (BIAS) {
#pragma unroll
        for (int e = 0; e < 2; e++)
#pragma unroll
          for (int c = 0; c < 2; c++)
            bv[e][c] = bf2f(reinterpret_cast<const short*>(&biases[side1][wid * 64])[32 * e + 2 * lo + c]);
      }
#pragma unroll
      for (int i = 0; i < 8; i++) {
        if (i * parts1 >= 8) continue;
        f32x2 cs[4] = {}, sn[4] = {};
        if (!is_v) {
#pragma unroll
          for (int r = 0; r < 4; r++) {
            const float* at = p.table + (long)turns[side1][gm0 - m1 + 16 * i + r] * D + d + 2 * lo;
            cs[r] = *reinterpret_cast<const f32x2*>(at);
            sn[r] = *reinterpret_cast<const f32x2*>(at + p.half);
          }
        }
#pragma unroll
        for (int r = 0; r < 4; r += 2) {
          unsigned w[2][2];                      // [half][row]
#pragma unroll
          for (int q = 0; q < 2; q++) {
#pragma unroll
            for (int e = 0; e < 2; e++)
              w[e][q] = pack2bf(acc[i][e][0][r + q] + bv[e][0], acc[i][e][1][r + q] + bv[e][1]);
            if (!is_v) {
              float o[2][2];
#pragma unroll
              for (int c = 0; c < 2; c++) {
                const float a = bf2f((short)(w[0][q] >> 16 * c)), b = bf2f((short)(w[1][q] >> 16 * c));
                o[0][c] = a * cs[r + q][c] - b * sn[r + q][c];
                o[1][c] = __builtin_fmaf(b, cs[r + q][c], a * sn[r + q][c]);
              }
#pragma unroll
              for (int e = 0; e < 2; e++) w[e][q] = pack2bf(o[e][0], o[e][1]);
            }
          }
          // neighbouring lanes exchange a row, so that each has 4 columns of one
          const int gm = gm0 + 16 * i + r + odd;
#pragma unroll
          for (int e = 0; e < 2; e++) {
            const unsigned mine = odd ? w[e][1] : w[e][0];
            const unsigned other =
                __builtin_amdgcn_mov_dpp(odd ? w[e][0] : w[e][1], 0xb1, 0xf, 0xf, true);
            if (gm < M1 && in)
              *reinterpret_cast<u32x2*>(to + gm * ld + e * p.half + 2 * lo - 2 * odd) =
                  odd ? u32x2{other, mine} : u32x2{mine, other};
          }
        }
      }
    } else {
      // neighbouring lanes exchange a row, so that each has 4 columns of one
      const bool odd = lo & 1;
      const int gn = n1 + wn / 2 + 2 * lo;
#pragma unroll
      for (int i = 0; i < 8; i++) {
        if (i * parts1 >= 8) continue;
#pragma unroll
        for (int r = 0; r < 4; r += 2) {
          float v[2][2];
          if constexpr (ACT == SILU_KEEP) {
            typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
            const int gm = gm0 + 16 * i + r + odd, gn4 = gn - 2 * odd;
            unsigned w[2][2];
#pragma unroll
            for (int e = 0; e < 2; e++) {
#pragma unroll
              for (int q = 0; q < 2; q++)
                w[e][q] = pack2bf(acc[i][e][0][r + q], acc[i][e][1][r + q]);
              const unsigned mine = odd ? w[e][1] : w[e][0];
              const unsigned other =
                  __builtin_amdgcn_mov_dpp(odd ? w[e][0] : w[e][1], 0xb1, 0xf, 0xf, true);
              if (gm < M1 && gn4 < p.N)
                __builtin_nontemporal_store(
                    odd ? u32x2{other, mine} : u32x2{mine, other},
                    reinterpret_cast<u32x2*>(p.kept + (long)gm * 2 * p.N + e * p.N + gn4));
            }
#pragma unroll
            for (int q = 0; q < 2; q++)
#pragma unroll
              for (int c = 0; c < 2; c++)
                v[q][c] = glu<ACT>(bf2f((short)(w[0][q] >> 16 * c)),
                                   bf2f((short)(w[1][q] >> 16 * c)));
          }
#pragma unroll
          for (int q = 0; q < 2 && ACT != SILU_KEEP; q++)
#pragma unroll
            for (int c = 0; c < 2; c++)
              v[q][c] = GROUPED ? act_silu(acc[i][0][c][r + q]) * acc[i][1][c][r + q] *
                                      scale_of(gm0 + 16 * i + r + q)
                                : glu<ACT>(acc[i][0][c][r + q], acc[i][1][c][r + q]);
          if (VEC) {
            typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
            const unsigned a = pack2bf(v[0][0], v[0][1]), b = pack2bf(v[1][0], v[1][1]);
            const unsigned mine = odd ? b : a;
            const unsigned other = __builtin_amdgcn_mov_dpp(odd ? a : b, 0xb1, 0xf, 0xf, true);
            const int gm = gm0 + 16 * i + r + odd, gn4 = gn - 2 * odd;
            if (gm < M1 && gn4 < p.N)
              __builtin_nontemporal_store(odd ? u32x2{other, mine} : u32x2{mine, other},
                                          reinterpret_cast<u32x2*>(row_of(gm) + gn4));
          } else {
#pragma unroll
            for (int q = 0; q < 2; q++)
#pragma unroll
              for (int c = 0; c < 2; c++)
                if (gm0 + 16 * i + r + q < M1 && gn + c < p.N)
                  row_of(gm0 + 16 * i + r + q)[gn + c] = f2bf(v[q][c]);
          }
        }
      }
    }
    if (!another) break;
    // a wave that stored less cannot count on its stores in the waits
    if (!VEC || parts1 > 1 || m1 + BIG > M1 || n1 + TN > p.N) wait_loads<0>();
  }
}

template <bool HAS_LORA, int BIAS, bool VEC, int ACT>
void launch_big(Big p) {
  const int cus = at::cuda::getCurrentDeviceProperties()->multiProcessorCount;
  constexpr int TN = big_columns(ACT);
  p.grid_m = (p.M + BIG - 1) / BIG;
  p.grid_n = (p.N + TN - 1) / TN;
  const int tiles = p.grid_m * p.grid_n, left = tiles % cus;
  p.parts = parts_of(left, cus);
  p.whole = p.parts > 1 ? tiles - left : tiles;
  p.units = p.whole + (tiles - p.whole) * p.parts;
  hipLaunchKernelGGL((gemm_big_kernel<HAS_LORA, BIAS, VEC, ACT>), dim3(std::min(p.units, cus)),
                     dim3(512), 0, c10::hip::getCurrentHIPStream(), p);
}

// Grouped products of whole steps of the depth, N and the strides of y multiples of 4: `most`
// tiles of rows at most.  A workgroup counts the groups' tiles at its start and finds the
// group of each as it comes to it; which rows of x and y they are is kept in LDS.  16
// experts of 1536 x 2240, 1000 rows each, gate and up 211 us (1050 TFLOP/s), down 100; in
// tiles of 128 that wait at a barrier a step 299 and 145.  The tiles left after whole rounds are
// divided as those of a single product, and a group's last tile takes as many rows as it has
// (64, 128 or all): 4 products of 2708 x 1536 x 1536 (264 tiles) 72 us, divided 63; the experts
// of 1536 x 2240 with 300 rows each 148 and 132 us, 677 300 and 286; the bits stay.  Silu is divided, as those have it,
// which takes 17 us of the 211: the bits are theirs, on which a router's near ties hang.
template <int ACT>
void launch_big_grouped(Big p, long most) {
  static_assert(ACT == NO_ACT || ACT == SILU_GLU, "silu alone is divided");
  const int cus = at::cuda::getCurrentDeviceProperties()->multiProcessorCount;
  constexpr int TN = ACT ? BIG / 2 : BIG;
  p.grid_n = (p.N + TN - 1) / TN;
  p.cus = cus;
  hipLaunchKernelGGL((gemm_big_kernel<false, NO_BIAS, true, ACT, true>),
                     dim3(std::min<long>(most * p.grid_n * 4, cus)), dim3(512), 0,
                     c10::hip::getCurrentHIPStream(), p);
}
