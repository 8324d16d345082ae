// Temperature / top-p token sampling over [B, V] bf16 or float32 logits.
// One workgroup of 1024 threads per row, which holds the whole row in registers
// (a CU's register file is 512 KB, a row of 151936 bf16 logits 304 KB) and reads
// it once:
//   1. row maximum
//   2. sum of exp(u), u = (l - max) / T, and its histogram over 32 bins of 1 nat
//   3. the bin in which the kept mass reaches top_p, refined into 32 parts once or
//      twice (no sort)
//   4. kept mass per thread + one block scan + inverse-CDF walk over the owner's
//      elements (counter-hash uniform: deterministic in (seed, step, row),
//      replay-safe via a device-side step counter for hipGraphs).
// Rows too long for the registers are read again for every pass.
//
// Few rows leave most CUs idle: sample_slices_kernel divides 1 and the sum of 2 among
// workgroups, and sample_row_kernel goes on with the row's few likely elements, or, where
// they are many, with a pass around the bin that a sample of the row names.
//
// A top-p of 1 keeps every token, which needs no bins and no row in registers: sample_all_kernel.
#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>

#include <type_traits>

#include "common.h"

#define SBLOCK 1024
#define SWAVES (SBLOCK / 64)
#define OWNERS 256     // the order of the categories: vectors of 8 elements, by index % OWNERS, then index
#define BINS 32
#define URANGE 32.0f   // the histogram covers u in [-URANGE, 0]; smaller ones fall into bin 0

template <typename LT> struct Vec8;
template <> struct Vec8<short> { s16x8 r; };
template <> struct Vec8<float> { f32x4 r[2]; };
DEVINL void load8(const short* p, Vec8<short>& v) { v.r = *reinterpret_cast<const s16x8*>(p); }
DEVINL void load8(const float* p, Vec8<float>& v) {
  v.r[0] = *reinterpret_cast<const f32x4*>(p);
  v.r[1] = *reinterpret_cast<const f32x4*>(p + 4);
}
DEVINL void fill8(Vec8<short>& v) {
#pragma unroll
  for (int j = 0; j < 8; j++) v.r[j] = (short)0xff80;   // -inf
}
DEVINL void fill8(Vec8<float>& v) {
#pragma unroll
  for (int j = 0; j < 4; j++) v.r[0][j] = v.r[1][j] = -INFINITY;
}
DEVINL void get8(const Vec8<short>& v, float* o) {
#pragma unroll
  for (int j = 0; j < 8; j++) o[j] = bf2f(v.r[j]);
}
DEVINL void get8(const Vec8<float>& v, float* o) {
#pragma unroll
  for (int j = 0; j < 8; j++) o[j] = v.r[j >> 2][j & 3];
}
// the compiler may not keep what an earlier pass made of v: unpacked, a row does
// not fit the registers
DEVINL void anew(Vec8<short>& v) { asm volatile("" : "+v"(v.r)); }
DEVINL void anew(Vec8<float>& v) { asm volatile("" : "+v"(v.r[0]), "+v"(v.r[1])); }
DEVINL float max8(const float* v) {
  float m = v[0];
#pragma unroll
  for (int j = 1; j < 8; j++) m = fmaxf(m, v[j]);
  return m;
}

// A row as its thread's vectors tid, tid + SBLOCK, ...: NV of them in registers,
// or (NV = 0) read anew by every pass.  The V % 8 last elements belong to the
// first threads, behind their vectors.
template <typename LT, int NV>
struct Row {
  const LT* p;
  int nvec, V;
  Vec8<LT> c[NV ? NV : 1];
  float most[NV ? NV : 1];      // each one's largest element

  DEVINL void load() {
    if (nvec == 0) {
#pragma unroll
      for (int k = 0; k < NV; k++) fill8(c[k]);
      return;
    }
#pragma unroll
    for (int k = 0; k < NV; k++)
      load8(p + 8L * min((int)threadIdx.x + SBLOCK * k, nvec - 1), c[k]);
#pragma unroll
    for (int k = 0; k < NV; k++)
      if ((int)threadIdx.x + SBLOCK * k >= nvec) fill8(c[k]);
  }
  // f(the largest of 8 logits)
  template <typename F> DEVINL void maxima(F f) {
    if constexpr (NV > 0) {
#pragma unroll
      for (int k = 0; k < NV; k++) {
        float v[8];
        anew(c[k]);
        get8(c[k], v);
        most[k] = max8(v);
        f(most[k]);
        __builtin_amdgcn_sched_barrier(0);
      }
    } else {
      vectors([&](int, const float* v) { f(max8(v)); });
    }
  }
  // f(first element's index, 8 logits, -inf where there are none)
  template <typename F> DEVINL void vectors(F f) {
    if constexpr (NV > 0) {
#pragma unroll
      for (int k = 0; k < NV; k++) {
        float v[8];
        anew(c[k]);
        get8(c[k], v);
        f(8 * (threadIdx.x + SBLOCK * k), v);
        __builtin_amdgcn_sched_barrier(0);     // registers for one vector at a time
      }
    } else {
      for (int i = threadIdx.x; i < nvec; i += SBLOCK) {
        Vec8<LT> w;
        load8(p + 8L * i, w);
        float v[8];
        get8(w, v);
        f(8 * i, v);
      }
    }
  }
  // of those only that some lane of the wave has an element in which is worth it
  template <typename W, typename F> DEVINL void vectors(W worth, F f) {
    if constexpr (NV > 0) {
#pragma unroll
      for (int k = 0; k < NV; k++) {
        if (!__any(worth(most[k]))) continue;
        float v[8];
        anew(c[k]);
        get8(c[k], v);
        f(v);
        __builtin_amdgcn_sched_barrier(0);
      }
    } else {
      vectors([&](int, const float* v) {
        if (__any(worth(max8(v)))) f(v);
      });
    }
  }
  DEVINL bool has_tail() const { return 8 * nvec + (int)threadIdx.x < V; }
  DEVINL float tail() const { return ldf(p + 8 * nvec + threadIdx.x); }
};

// Histogram columns are private to a lane of a wave, so that the adds meet no
// other thread's: conflict-free, and in a fixed order.  (A histogram of 32
// registers per thread costs 32 selects per element, which was most of the
// kernel; one shared by the block serialises on its bins.)
struct Scratch {
  float hist[SWAVES][BINS][64];
  float red[SWAVES];
  float mass[BINS];
  float own[SBLOCK];
  float lo, above, excl;
  int index[SWAVES];
  int done, found, owner;
};

DEVINL void clear_hist(Scratch& s) {
  f32x4* h = reinterpret_cast<f32x4*>(s.hist);
  for (int i = threadIdx.x; i < SWAVES * BINS * 16; i += SBLOCK) h[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  __syncthreads();
}
DEVINL void add_hist(Scratch& s, float bin, float e) {
  const int b = max(0, min(BINS - 1, (int)bin));
  s.hist[threadIdx.x >> 6][b][threadIdx.x & 63] += e;
}
// The first wave finds the highest bin at which the mass from the top, `above`
// included, reaches `target` (or bin 0), and moves lo, above and done there.
DEVINL void choose_bin(Scratch& s, float above, float target, float lo, float width, float S,
                       bool refined) {
  __syncthreads();
  {
    const int b = threadIdx.x >> 5, l = threadIdx.x & 31;   // 32 threads per bin
    float x = 0.f;
#pragma unroll 4
    for (int w = 0; w < SWAVES; w++) x += s.hist[w][b][l] + s.hist[w][b][l + 32];
#pragma unroll
    for (int off = 16; off > 0; off >>= 1) x += __shfl_xor(x, off);
    if (l == 0) s.mass[b] = x;
  }
  __syncthreads();
  if (threadIdx.x < 64) {
    const int lane = threadIdx.x;
    const float h = lane < BINS ? s.mass[BINS - 1 - lane] : 0.f;   // from the top down
    float incl = h;
#pragma unroll
    for (int off = 1; off < BINS; off <<= 1) {
      const float x = __shfl_up(incl, off);
      if (lane >= off) incl += x;
    }
    const unsigned long long hit = __ballot(lane < BINS && above + incl >= target);
    const int at = hit ? __ffsll((unsigned long long)hit) - 1 : BINS - 1;
    if (lane == at) {
      s.lo = lo + (float)(BINS - 1 - at) * width;
      s.above = above + (incl - h);
      // over-keeping a sliver of the boundary bin changes the nucleus by < 2% of S
      s.done = refined && h <= 0.02f * S;
    }
  }
  __syncthreads();
}

// largest element and its lowest index (0 where nothing is above -inf)
template <int BLOCK, typename LT>
DEVINL int row_argmax(const LT* __restrict__ p, int V, float& best, float* red, int* index) {
  float top = -INFINITY;
  int at = 0;
#pragma unroll 4
  for (int i = threadIdx.x; i < V / 8; i += BLOCK) {
    float v[8];
    ldv<8>(p + 8L * i, v);
#pragma unroll
    for (int j = 0; j < 8; j++)
      if (v[j] > top) { top = v[j]; at = 8 * i + j; }
  }
  const int t = V / 8 * 8 + threadIdx.x;
  if (t < V && ldf(p + t) > top) { top = ldf(p + t); at = t; }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const float top2 = __shfl_xor(top, off);
    const int at2 = __shfl_xor(at, off);
    if (top2 > top || (top2 == top && at2 < at)) { top = top2; at = at2; }
  }
  if ((threadIdx.x & 63) == 0) { red[threadIdx.x >> 6] = top; index[threadIdx.x >> 6] = at; }
  __syncthreads();
  top = red[0];
  at = index[0];
  for (int w = 1; w < BLOCK / 64; w++)
    if (red[w] > top || (red[w] == top && index[w] < at)) { top = red[w]; at = index[w]; }
  __syncthreads();
  best = top;
  return at;
}

// temperature 0: the most likely token, and its logprob under the softmax at T = 1.
// A kernel of its own, because several rows to a CU hide each other's loads, which
// the other's histogram leaves no LDS for.
template <typename LT, int BLOCK>
__global__ __launch_bounds__(BLOCK)
void sample_greedy_kernel(const LT* __restrict__ logits, long* __restrict__ out,
                          float* __restrict__ out_lp, int V) {
  __shared__ float red[BLOCK / 64];
  __shared__ int index[BLOCK / 64];
  const long row = blockIdx.x;
  const LT* p = logits + row * (long)V;
  float top;
  const int at = row_argmax<BLOCK>(p, V, top, red, index);
  if (threadIdx.x == 0) out[row] = at;
  if (!out_lp) return;
  float se = 0.f;
#pragma unroll 4
  for (int i = threadIdx.x; i < V / 8; i += BLOCK) {
    float v[8];
    ldv<8>(p + 8L * i, v);
#pragma unroll
    for (int j = 0; j < 8; j++) se += __expf(v[j] - top);
  }
  const int t = V / 8 * 8 + threadIdx.x;
  if (t < V) se += __expf(ldf(p + t) - top);
  se = block_sum<BLOCK>(se, red);
  if (threadIdx.x == 0) out_lp[row] = ldf(p + at) - (top + __logf(se));
}

template <typename LT, int NV>
__global__ __launch_bounds__(SBLOCK)
void sample_topp_kernel(const LT* __restrict__ logits,
                        long* __restrict__ out,
                        float* __restrict__ out_lp,  // nullable
                        int V, float temperature, float top_p,
                        unsigned long long seed,
                        unsigned long long step_imm,
                        const long* __restrict__ step_ptr) {
  __shared__ Scratch s;
  const unsigned long long step = step_imm + (step_ptr ? (unsigned long long)*step_ptr : 0);
  const long row = blockIdx.x;
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  Row<LT, NV> r;
  r.p = logits + row * (long)V;
  r.nvec = V / 8;
  r.V = V;
  r.load();

  // ---- 1: row maximum ---------------------------------------------------
  float top = -INFINITY;
  r.maxima([&](float m) { top = fmaxf(top, m); });
  if (r.has_tail()) top = fmaxf(top, r.tail());
  top = block_max<SBLOCK>(top, s.red);

  const float invT = temperature > 0.f ? 1.f / temperature : 1.f;
  const float M = top * invT;           // max of temperature-scaled logits

  // ---- 2: sum and coarse histogram ---------------------------------------
  clear_hist(s);
  float sum = 0.f;
  auto coarse = [&](float l) {
    const float u = l * invT - M, e = __expf(u);
    sum += e;
    add_hist(s, u + URANGE, e);
  };
  r.vectors([&](int, const float* v) {
#pragma unroll
    for (int j = 0; j < 8; j++) coarse(v[j]);
  });
  if (r.has_tail()) coarse(r.tail());
  const float S = block_sum<SBLOCK>(sum, s.red);
  const float target = top_p * S;
  choose_bin(s, 0.f, target, -URANGE, 1.f, S, false);

  // ---- 3: refine the boundary bin until it is narrow (1/1024 nat) or holds
  // negligible mass; vectors without an element in it are passed over ---------
  float width = 1.f;
  for (int it = 0; it < 2 && !s.done; it++) {
    const float lo = s.lo, above = s.above, scale = BINS / width;
    clear_hist(s);
    auto fine = [&](float l) {
      const float u = l * invT - M;
      if (u >= lo && u < lo + width) add_hist(s, (u - lo) * scale, __expf(u));
    };
    r.vectors([&](float most) { return most * invT - M >= lo; }, [&](const float* v) {
#pragma unroll
      for (int j = 0; j < 8; j++) fine(v[j]);
    });
    if (r.has_tail()) fine(r.tail());
    choose_bin(s, above, target, lo, width / BINS, S, true);
    width /= BINS;
  }
  const float lowest = s.lo;

  // ---- 4: kept mass, scan over the owners, walk --------------------------
  auto kept = [&](float l) {
    const float u = l * invT - M;
    return u >= lowest ? __expf(u) : 0.f;
  };
  float own = 0.f;
  r.vectors([&](float most) { return most * invT - M >= lowest; }, [&](const float* v) {
#pragma unroll
    for (int j = 0; j < 8; j++) own += kept(v[j]);
  });
  if (r.has_tail()) own += kept(r.tail());
  s.own[tid] = own;
  if (tid == 0) { s.owner = OWNERS; s.found = -1; }
  __syncthreads();
  own = 0.f;
  if (tid < OWNERS) {
#pragma unroll
    for (int k = 0; k < SBLOCK / OWNERS; k++) own += s.own[tid + OWNERS * k];
  }
  float incl = own;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const float x = __shfl_up(incl, off);
    if (lane >= off) incl += x;
  }
  if (lane == 63) s.red[wid] = incl;
  __syncthreads();
  float base = 0.f, total = 0.f;
  for (int w = 0; w < OWNERS / 64; w++) {
    if (w < wid) base += s.red[w];
    total += s.red[w];
  }
  const float goal = hash_uniform(seed, step, (unsigned long long)row) * total;
  const float excl = base + incl - own;
  // rounding may leave two at a border: the first
  if (tid < OWNERS && own > 0.f && goal >= excl && goal < excl + own) atomicMin(&s.owner, tid);
  __syncthreads();
  if (tid == s.owner) s.excl = excl;
  __syncthreads();
  if (wid == 0 && s.owner < OWNERS) {
    // the owner's vectors in order, 64 at a time, one per lane
    float acc = s.excl;
    bool found = false;
    for (int i0 = s.owner; i0 < r.nvec && !found; i0 += OWNERS * 64) {
      const int i = i0 + OWNERS * lane;
      float e[8], m = 0.f;
      Vec8<LT> w;
      if (i < r.nvec) load8(r.p + 8L * i, w);
      else fill8(w);
      get8(w, e);
#pragma unroll
      for (int j = 0; j < 8; j++) {
        e[j] = kept(e[j]);
        m += e[j];
      }
      float upto = m;
#pragma unroll
      for (int off = 1; off < 64; off <<= 1) {
        const float x = __shfl_up(upto, off);
        if (lane >= off) upto += x;
      }
      const unsigned long long hit = __ballot(m > 0.f && goal < acc + upto);
      if (hit) {
        found = true;
        if (lane == __ffsll((unsigned long long)hit) - 1) {
          float at = acc + (upto - m);
          int last = -1, pick = -1;
#pragma unroll
          for (int j = 0; j < 8; j++) {
            at += e[j];
            if (e[j] > 0.f) last = j;
            if (pick < 0 && e[j] > 0.f && goal < at) pick = j;
          }
          s.found = 8 * i + (pick >= 0 ? pick : last);
        }
      }
      acc += __shfl(upto, 63);
    }
    const int t = 8 * r.nvec + s.owner;
    if (!found && lane == 0 && t < V && goal < acc + kept(ldf(r.p + t))) s.found = t;
  }
  __syncthreads();
  int pick = s.found;
  if (pick < 0) {                       // rounding: no element crosses the goal
    float best;
    pick = row_argmax<SBLOCK>(r.p, V, best, s.red, s.index);
  }
  if (tid == 0) {
    out[row] = pick;
    // logprob of the chosen token under the temperature-scaled softmax
    // (matches the scoring pass's logits/temperature quirk, grpo_trainer.py:547)
    if (out_lp) out_lp[row] = ldf(r.p + pick) * invT - (M + __logf(S));
  }
}

// A part of a row may hold nothing but a mask, -1e10 or the type's lowest value, and so far from 0
// top / T is no subtrahend of l / T: its rounding alone is a large exponent, or it is -inf.  There
// the exponents are (l - top) / T.
DEVINL bool far_below(float top, float invT) { return top * invT < -1e6f && top > -INFINITY; }

// Every element once, by workgroups of 256 threads, 8 vectors a thread: `part` [B, slices],
// a slice's largest logit and its sum of exp((l - that) / T), and `runs` [B, RBLOCK, RUN], the
// vectors' largest elements, where a thread of the row's workgroup finds a run of RUN vectors
// of one owner next to each other (half the owner's).  A slice without anything above -inf has a sum of 0, or a
// not-a-number if it holds one.
constexpr int RBLOCK = 512, RWAVES = RBLOCK / 64;
constexpr int SLICE_VECS = 8, SLICE = OWNERS * SLICE_VECS;
template <typename LT, int RUN>
__global__ __launch_bounds__(OWNERS)
void sample_slices_kernel(const LT* __restrict__ logits, float2* __restrict__ part,
                          LT* __restrict__ runs, int V, float invT) {
  static_assert(RUN % SLICE_VECS == 0, "a slice's vectors of an owner are of one run");
  __shared__ float red[OWNERS / 64];
  const long row = blockIdx.y;
  const int nvec = V / 8, at = blockIdx.x * SLICE + threadIdx.x;
  const LT* p = logits + row * (long)V;
  Vec8<LT> c[SLICE_VECS];
#pragma unroll
  for (int k = 0; k < SLICE_VECS; k++)
    load8(p + 8L * min(at + OWNERS * k, nvec - 1), c[k]);
  // the last elements belong to the last slice
  const int t = 8 * nvec + threadIdx.x;
  const float tail = blockIdx.x == gridDim.x - 1 && t < V ? ldf(p + t) : -INFINITY;
  float top = tail, m[SLICE_VECS];
#pragma unroll
  for (int k = 0; k < SLICE_VECS; k++) {
    if (at + OWNERS * k >= nvec) fill8(c[k]);
    float v[8];
    get8(c[k], v);
    m[k] = max8(v);
    top = fmaxf(top, m[k]);
  }
  const int j = blockIdx.x * SLICE_VECS;
  stv<SLICE_VECS>(runs + ((row * OWNERS + threadIdx.x) * 2 + j / RUN) * RUN + j % RUN, m);
  top = block_max<OWNERS>(top, red);
  float sum = 0.f;
  const auto add = [&](auto e) {
    sum = e(tail);
#pragma unroll
    for (int k = 0; k < SLICE_VECS; k++) {
      float v[8];
      get8(c[k], v);
#pragma unroll
      for (int j = 0; j < 8; j++) sum += e(v[j]);
    }
  };
  const float M = top == -INFINITY ? 0.f : top * invT;
  if (far_below(top, invT)) add([&](float l) { return __expf((l - top) * invT); });
  else add([&](float l) { return __expf(l * invT - M); });
  sum = block_sum<OWNERS>(sum, red);
  if (threadIdx.x == 0) part[row * gridDim.x + blockIdx.x] = float2{top, sum};
}

// inclusive sums over the lanes before
template <typename T>
DEVINL T lanes_before(T v) {
  static_assert(sizeof(T) == 4, "");
  auto shift = [&](auto ctrl) {
    v += __builtin_bit_cast(T, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v),
                                                           decltype(ctrl)::value, 0xf, 0xf, true));
  };
  shift(std::integral_constant<int, 0x111>{});    // row_shr:1, 2, 4, 8
  shift(std::integral_constant<int, 0x112>{});
  shift(std::integral_constant<int, 0x114>{});
  shift(std::integral_constant<int, 0x118>{});
  auto of = [&](int lane) {
    return __builtin_bit_cast(T, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), lane));
  };
  const T a = of(15), b = a + of(31), c = b + of(47);
  const int r = (threadIdx.x & 63) >> 4;
  return r == 0 ? v : v + (r == 1 ? a : r == 2 ? b : c);
}
template <typename T>
DEVINL T of_lane(T v, int lane) {     // a lane that all agree on
  return __builtin_bit_cast(T, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), lane));
}

// The row's workgroup behind sample_slices_kernel, with the same bins, thresholds, categories
// and order of them as sample_topp_kernel.  Bound by a chain of some 15 dependent steps where
// the nucleus is small (8 rows of 151936: 11.2 us with the slices, of which each kernel's
// start and first loads are half; one kernel 26.0), and else by reading, adding and writing
// back the columns of the bins on one CU.
constexpr int LIKELY = 4096;
struct RowScratch {
  union {
    float hist[RWAVES][2 * BINS + 2][64];   // columns private to a lane, as Scratch's
    struct {
      float u[LIKELY];
      int id[LIKELY];
    } likely;
  };
  // Masses of bins in multiples of 2^-42: exact for an exp(u) of at least exp(-12), which has
  // 24 bits, whatever the order; and integers are added up in LDS much faster than floats
  // (67 and 3073 cycles for 16 waves; reading, adding and writing back takes 130).
  unsigned long long exact[BINS];
  float bin[2 * BINS], red[RWAVES];
  int count[RWAVES];
  int pick;
};
DEVINL unsigned long long exactly(float e) { return (unsigned long long)(e * 0x1p42f); }

// Of 64 lanes' masses, from the top: the first lane at which `above` and they reach the target
// (-1: none), and the mass above it.
DEVINL int reach(float mass, float above, float target, float& before) {
  const float incl = lanes_before(mass);
  const unsigned long long hit = __ballot(above + incl >= target);
  const int at = hit ? __ffsll(hit) - 1 : -1;
  before = above + of_lane(incl - mass, max(at, 0));
  return at;
}
// the sum over the lanes and waves ahead, for all threads, and that of all
template <typename T>
DEVINL T block_before(T v, T* scratch, T& total) {
  const int wid = threadIdx.x >> 6;
  const T incl = lanes_before(v);
  if ((threadIdx.x & 63) == 63) scratch[wid] = incl;
  __syncthreads();
  T base{};
  total = T{};
#pragma unroll
  for (int w = 0; w < RWAVES; w++) {
    if (w < wid) base += scratch[w];
    total += scratch[w];
  }
  __syncthreads();
  return base + incl - v;
}

template <typename LT, int RUN>
__global__ __launch_bounds__(RBLOCK)
void sample_row_kernel(const LT* __restrict__ logits, long* __restrict__ out,
                       float* __restrict__ out_lp, int V, float invT, float top_p,
                       unsigned long long seed, unsigned long long step_imm,
                       const long* __restrict__ step_ptr, const float2* __restrict__ part,
                       const LT* __restrict__ runs, int slices) {
  __shared__ __attribute__((aligned(16))) RowScratch s;
  const unsigned long long step = step_imm + (step_ptr ? (unsigned long long)*step_ptr : 0);
  const long row = blockIdx.x;
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6, nvec = V / 8;
  const LT* p = logits + row * (long)V;
  const float uniform = of_lane(hash_uniform(seed, step, (unsigned long long)row), 0);

  // Two threads an owner, so that what they find has the order of the categories; the
  // owner's element of the V % 8 last ones behind its vectors.
  const int owner = tid >> 1, first = owner + OWNERS * RUN * (tid & 1);
  const int t = (tid & 1) ? 8 * nvec + owner : V;
  float most[RUN];
#pragma unroll
  for (int k = 0; k < RUN; k += 8) ldv<8>(runs + (row * RBLOCK + tid) * RUN + k, most + k);
  const float tail = t < V ? ldf(p + t) : -INFINITY;
  const float2 w = lane < slices ? part[row * slices + lane] : float2{-INFINITY, 0.f};
  const float top = wave_max(w.x);
  const float M = of_lane(top * invT, 0);
  const float S = of_lane(wave_sum(w.x == top ? w.y : w.y * __expf(w.x * invT - M)), 0);
  const float target = top_p * S;
  const auto scaled = [&](float l) { return l * invT - M; };
#pragma unroll
  for (int k = 0; k < RUN; k++)       // past the row's end is whatever the memory held
    most[k] = first + OWNERS * k < nvec ? scaled(most[k]) : -INFINITY;

  // logprob of the chosen token under the temperature-scaled softmax
  // (matches the scoring pass's logits/temperature quirk, grpo_trainer.py:547)
  const auto put = [&](int pick) {
    out[row] = pick;
    if (out_lp) out_lp[row] = ldf(p + pick) * invT - (M + __logf(S));
  };
  // f(8 u, the first one's index) of this thread's vectors with one at `least` or above, and
  // of the tail's element, with -inf behind it
  const auto each = [&](float least, auto f) {
    unsigned long long ones = 0;
#pragma unroll
    for (int k = 0; k < RUN; k++) ones |= (most[k] >= least ? 1ull : 0ull) << k;
    while (__any(ones != 0)) {
      constexpr int FEW = 4;           // loads in flight
      Vec8<LT> c[FEW];
      int at[FEW];
#pragma unroll
      for (int i = 0; i < FEW; i++) {
        at[i] = ones ? first + OWNERS * (__ffsll(ones) - 1) : -1;
        ones &= ones - 1;
        fill8(c[i]);
        if (at[i] >= 0) load8(p + 8L * at[i], c[i]);
      }
#pragma unroll
      for (int i = 0; i < FEW; i++) {
        if (!__any(at[i] >= 0)) break;
        float v[8];
        get8(c[i], v);
#pragma unroll
        for (int j = 0; j < 8; j++) v[j] = scaled(v[j]);
        f(v, 8 * at[i]);
      }
    }
    float v[8];
#pragma unroll
    for (int j = 0; j < 8; j++) v[j] = j ? -INFINITY : scaled(tail);
    if (__any(t < V)) f(v, t);
  };

  // ---- few likely elements ------------------------------------------------
  // A language model's logits fall with the rank's logarithm: few are within some nats of
  // the maximum and hold the nucleus, 8 at a temperature of 0.7 and 12 at 1.  `upper`: what
  // is at `from` or above.
  float from = 0.f, upper = 0.f;
  bool few = S > 0.f;
  for (float near = 8.f; few && near <= 12.f; near += 4.f) {
    // rows of many are known by their vectors
    int n = 0, total;
#pragma unroll
    for (int k = 0; k < RUN; k++) n += most[k] >= -near;
    block_before(n, s.count, total);
    if (total > LIKELY) break;
    n = 0;
    each(-near, [&](const float* u, int) {
#pragma unroll
      for (int j = 0; j < 8; j++) n += u[j] >= -near;
    });
    int at = block_before(n, s.count, total);
    if (total > LIKELY) break;
    each(-near, [&](const float* u, int i) {
#pragma unroll
      for (int j = 0; j < 8; j++)
        if (u[j] >= -near) {
          s.likely.u[at] = u[j];
          s.likely.id[at++] = i + j;
        }
    });
    // the bin at which the mass reaches the target, and its refinements
    float lo = -URANGE, width = 1.f, above = 0.f;
    bool done = false;
    for (int it = 0; it < 3 && !done; it++) {
      if (tid < BINS) s.exact[tid] = 0;
      __syncthreads();
      const float scale = 1.f / width;
      for (int i = tid; i < total; i += RBLOCK) {
        const float u = s.likely.u[i];
        if (it == 0 || (u >= lo && u < lo + BINS * width))
          atomicAdd(&s.exact[max(0, min(BINS - 1, (int)((u - lo) * scale)))], exactly(__expf(u)));
      }
      __syncthreads();
      const float mass = lane < BINS ? (float)s.exact[BINS - 1 - lane] * 0x1p-42f : 0.f;
      __syncthreads();
      float before;
      const int hit = reach(mass, above, target, before);
      const int at = hit < 0 || hit >= BINS ? BINS - 1 : hit;
      if (it == 0 && !(hit >= 0 && lo + (float)(BINS - 1 - at) >= -near)) {
        from = -near;
        upper = wave_sum(lane < (int)near ? mass : 0.f);
        lo = -INFINITY;
        break;
      }
      above = hit < 0 ? above + wave_sum(lane < BINS - 1 ? mass : 0.f) : before;
      lo += (float)(BINS - 1 - at) * width;
      // over-keeping a sliver of the boundary bin changes the nucleus by < 2% of S
      done = it > 0 && of_lane(mass, at) <= 0.02f * S;
      width /= BINS;
    }
    if (lo == -INFINITY) continue;
    const auto kept = [&](int i) {
      const float u = s.likely.u[i];
      return u >= lo ? __expf(u) : 0.f;
    };
    const int share = (total + RBLOCK - 1) / RBLOCK, i0 = min(tid * share, total);
    const int i1 = min(i0 + share, total);
    float own = 0.f, all;
    for (int i = i0; i < i1; i++) own += kept(i);
    if (tid == 0) s.pick = RBLOCK;
    float sum = block_before(own, s.red, all);
    const float goal = uniform * all;
    // rounding may leave two at a border: the first
    const bool mine = own > 0.f && goal >= sum && goal < sum + own;
    if (mine) atomicMin(&s.pick, tid);
    __syncthreads();
    const int chosen = s.pick;
    if (chosen == RBLOCK) break;        // rounding: none
    if (tid == chosen) {
      int pick = -1;
      for (int i = i0; i < i1; i++) {
        const float e = kept(i);
        sum += e;
        if (e > 0.f) {
          pick = s.likely.id[i];
          if (goal < sum) break;
        }
      }
      put(pick);
    }
    return;
  }

  // ---- many: a pass over two bins at a time, which leaves every thread the mass of each of
  // their refined bins (as hist's columns), and so its own kept mass -----------
  const auto clear = [&](int bins) {
    for (int i = tid; i < RWAVES * bins * 16; i += RBLOCK)
      reinterpret_cast<f32x4*>(&s.hist[i / (bins * 16)][0][0])[i % (bins * 16)] = f32x4{};
    __syncthreads();
  };
  const auto sum_bins = [&](int from) {         // of all columns, 8 threads a bin
    __syncthreads();
    float x = 0.f;
#pragma unroll
    for (int w = 0; w < RWAVES; w++)
#pragma unroll
      for (int c = 0; c < 8; c++) x += s.hist[w][from + (tid >> 3)][8 * c + (tid & 7)];
#pragma unroll
    for (int off = 4; off > 0; off >>= 1) x += __shfl_xor(x, off);
    if ((tid & 7) == 0) s.bin[tid >> 3] = x;
    __syncthreads();
  };
  const auto columns = [&](int a, int b) {      // this lane's, of bins [a, b)
    float x = 0.f;
    for (int i = a; i < b; i++) x += s.hist[wid][i][lane];
    return x;
  };
  float own = 0.f, lowest = -URANGE;
  if (few) {       // S is a number
    __syncthreads();
    clear(BINS);
    {
      Vec8<LT> c;
      float v[8];
      load8(p + 8L * ((long)tid * nvec / RBLOCK), c);
      get8(c, v);
#pragma unroll
      for (int j = 0; j < 8; j++) {
        const float u = scaled(v[j]);
        if (u < from || from == 0.f)
          s.hist[wid][max(0, min(BINS - 1, (int)(u + URANGE)))][lane] += __expf(u);
      }
    }
    sum_bins(0);
    // bins from the top; what is left of S is divided as the sample is
    const float some = lane < BINS ? s.bin[BINS - 1 - lane] : 0.f, rest = wave_sum(some);
    const float mass = rest > 0.f ? some * ((S - upper) / rest) : 0.f;
    float before;
    const int at = reach(mass, upper, target, before);
    const float in = of_lane(mass, max(at, 0));
    float hi = at < 0 ? 2.f - URANGE : target - before < 0.5f * in ? 1.f - at : (float)-at;
    hi = fmaxf(fminf(hi, 0.f), 2.f - URANGE);
    float A, m1, m2;
    for (int moved = 0;;) {
      __syncthreads();
      clear(2 * BINS + 1);
      const float bottom = hi - 2.f;
      own = 0.f;
      // In pairs, whose columns are read before either is written: half the reads' latency,
      // which is what the pass takes.  Elements of neither bin go to one below or above, for
      // asking whether a wave has others takes more: 64 flat rows of 151936 48.2 us so, 44.8 now.
      // The bin by u's floor, which is exact, as kept's comparison is: u - bottom is rounded, and
      // an element just below a bin's upper border would be in the next.
      const int below = (int)bottom * BINS - 1;
      each(bottom, [&](const float* u, int) {
#pragma unroll
        for (int j = 0; j < 8; j += 2) {
          float e[2];
          int k[2];
#pragma unroll
          for (int i = 0; i < 2; i++) {
            e[i] = __expf(u[j + i]);
            own += u[j + i] >= hi ? e[i] : 0.f;
            k[i] = (int)floorf(__builtin_amdgcn_fmed3f(u[j + i] * BINS, below,
                                                       below + 2.f * BINS + 1.f)) - below;
          }
          float *h0 = &s.hist[wid][k[0]][lane], *h1 = &s.hist[wid][k[1]][lane];
          const float x = *h0 + e[0], y = *h1;
          *h0 = x;
          *h1 = (k[0] == k[1] ? x : y) + e[1];
        }
      });
      sum_bins(1);
      block_before(own, s.red, A);
      m2 = wave_sum(lane < BINS ? s.bin[lane] : 0.f);
      m1 = wave_sum(lane < BINS ? s.bin[BINS + lane] : 0.f);
      if (A >= target && hi < 0.f && moved >= 0) {
        hi = fminf(hi + 2.f, 0.f);
        moved = 1;
      } else if (A + (m1 + m2) < target && bottom > -URANGE && moved <= 0) {
        hi = fmaxf(bottom, 2.f - URANGE);
        moved = -1;
      } else {
        break;
      }
    }
    const int b = A + m1 >= target ? BINS : 0;        // the upper of the two, or the lower
    if (!b) own += columns(1 + BINS, 1 + 2 * BINS);
    lowest = hi - (b ? 1.f : 2.f);
    // the maximum itself is of no refined bin
    float above = lowest == -1.f ? 0.f : b ? A : A + m1;
    const float x = lane < BINS ? s.bin[b + BINS - 1 - lane] : 0.f;
    int fine = reach(x, above, target, before);
    if (fine < 0 || fine >= BINS) {
      fine = BINS - 1;
      before = above + wave_sum(lane < fine ? x : 0.f);
    }
    above = before;
    fine = BINS - 1 - fine;
    lowest += fine * (1.f / BINS);
    own += columns(1 + b + fine + 1, 1 + b + BINS);
    // over-keeping a sliver of the boundary bin changes the nucleus by < 2% of S
    if (s.bin[b + fine] <= 0.02f * S) {
      own += s.hist[wid][1 + b + fine][lane];
    } else {
      __syncthreads();
      clear(BINS);
      const float lo = lowest;
      const int first_bin = (int)(lo * (BINS * BINS));
      each(lo, [&](const float* u, int) {
#pragma unroll
        for (int j = 0; j < 8; j++)
          if (u[j] >= lo && u[j] < lo + 1.f / BINS)
            s.hist[wid][(int)floorf(u[j] * (BINS * BINS)) - first_bin][lane] += __expf(u[j]);
      });
      sum_bins(0);
      const float y = lane < BINS ? s.bin[BINS - 1 - lane] : 0.f;
      fine = reach(y, above, target, before);
      fine = fine < 0 || fine >= BINS ? 0 : BINS - 1 - fine;
      lowest += fine * (1.f / (BINS * BINS));
      own += columns(fine, BINS);
    }
  } else {
    each(lowest, [&](const float* u, int) {
#pragma unroll
      for (int j = 0; j < 8; j++) own += u[j] >= lowest ? __expf(u[j]) : 0.f;
    });
  }

  // ---- scan and walk ---------------------------------------------------------
  const auto kept = [&](float u) { return u >= lowest ? __expf(u) : 0.f; };
  float all;
  if (tid == 0) s.pick = RBLOCK;
  const float sum = block_before(own, s.red, all), goal = uniform * all;
  if (own > 0.f && goal >= sum && goal < sum + own) atomicMin(&s.pick, tid);
  __syncthreads();
  const int chosen = s.pick;
  if (tid == chosen) s.bin[0] = sum;
  __syncthreads();
  if (tid == 0) s.pick = -1;
  __syncthreads();
  if (wid == 0 && chosen < RBLOCK) {
    // its vectors in order, one per lane, and the tail's element in the last
    static_assert(RUN < 64, "a run and one");
    const int run = (chosen >> 1) + OWNERS * RUN * (chosen & 1);
    const int i = run + OWNERS * lane, last = (chosen & 1) ? 8 * nvec + (chosen >> 1) : V;
    Vec8<LT> c;
    fill8(c);
    if (lane < RUN && i < nvec) load8(p + 8L * i, c);
    float e[8], m = 0.f;
    get8(c, e);
    if (lane == RUN && last < V) e[0] = ldf(p + last);
#pragma unroll
    for (int j = 0; j < 8; j++) {
      e[j] = kept(scaled(e[j]));
      m += e[j];
    }
    const float base = s.bin[0] + lanes_before(m) - m;
    const unsigned long long hit = __ballot(m > 0.f && goal < base + m);
    const unsigned long long any = __ballot(m > 0.f);
    // rounding may leave the goal behind all of them: the last
    const int owner = hit ? __ffsll(hit) - 1 : any ? 63 - __clzll(any) : -1;
    if (lane == owner) {
      float at = base;
      int pick = -1;
#pragma unroll
      for (int j = 0; j < 8; j++) {
        if (e[j] > 0.f && !(pick >= 0 && goal < at)) pick = lane == RUN ? last : 8 * i + j;
        at += e[j];
      }
      s.pick = pick;
    }
  }
  __syncthreads();
  int pick = s.pick;
  if (pick < 0) {                     // nothing is above -inf
    float best;
    pick = row_argmax<RBLOCK>(p, V, best, s.red, s.count);
  }
  if (tid == 0) put(pick);
}

// ------------------------------------------------------ top-p of 1: no bins
// Every token stays: a maximum and the owners' masses are all that sampling needs, in one pass
// that keeps no row.  A workgroup of a thread to an owner takes a row, or a slice of it where
// these are fewer than 2048, which fill the CUs with waves; a second kernel then adds up the
// slices' masses.  Bound by reading the logits (2048 rows of 151936: 113 us, 5.5 TB/s), for few
// rows by two launches and their chains of latencies.  bf16 at T = 1, through the bins / so, us:
//   151936   1 row 36.7 / 8.8   64 44.2 / 12.8   512 99.5 / 32.4   2048 371 / 113
//   32768    1 row 14.7 / 8.2   64 16.2 / 8.4    512 32.6 / 13.5   2048 121 / 24.3
//   1000     1 row 12.2 / 5.1   64 13.0 / 5.6    512 25.5 / 6.0    2048 94 / 8.9
// 32 bits of 151936: 64 rows 54.3 / 14.5, 2048 679 / 207.
constexpr int ALL_VECS = 4;       // of a thread, asked for together

struct PickScratch {
  float red[OWNERS / 64], excl;
  int index[OWNERS / 64], owner, found;
};

// A category by the owners' masses exp(l / T - top / T), of which each thread has one, and its
// log-probability.
template <typename LT>
DEVINL void pick_of_all(PickScratch& s, const LT* __restrict__ p, int V, float invT, float top,
                        float own, float uniform, long* __restrict__ out,
                        float* __restrict__ out_lp) {
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6, nvec = V / 8;
  const float M = top * invT;
  float incl = own;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const float x = __shfl_up(incl, off);
    if (lane >= off) incl += x;
  }
  if (lane == 63) s.red[wid] = incl;
  if (tid == 0) { s.owner = OWNERS; s.found = -1; }
  __syncthreads();
  float base = 0.f, total = 0.f;
#pragma unroll
  for (int w = 0; w < OWNERS / 64; w++) {
    if (w < wid) base += s.red[w];
    total += s.red[w];
  }
  const float goal = uniform * total, excl = base + incl - own;
  // rounding may leave two at a border: the first
  if (own > 0.f && goal >= excl && goal < excl + own) atomicMin(&s.owner, tid);
  __syncthreads();
  if (tid == s.owner) s.excl = excl;
  __syncthreads();
  if (wid == 0 && s.owner < OWNERS) {
    // the owner's vectors in order, 64 at a time, one per lane; behind them its last element
    float acc = s.excl;
    int last = -1;                  // of a mass, should rounding let no element cross the goal
    bool found = false;
    for (int i0 = s.owner; i0 < nvec && !found; i0 += OWNERS * 64) {
      const int i = i0 + OWNERS * lane;
      float e[8], m = 0.f;
      Vec8<LT> w;
      if (i < nvec) load8(p + 8L * i, w);
      else fill8(w);
      get8(w, e);
#pragma unroll
      for (int j = 0; j < 8; j++) {
        e[j] = __expf(e[j] * invT - M);
        m += e[j];
      }
      float upto = m;
#pragma unroll
      for (int off = 1; off < 64; off <<= 1) {
        const float x = __shfl_up(upto, off);
        if (lane >= off) upto += x;
      }
      const unsigned long long hit = __ballot(m > 0.f && goal < acc + upto);
      const unsigned long long some = __ballot(m > 0.f);
      found = hit != 0;
      if (some) {
        const int of = found ? __ffsll(hit) - 1 : 63 - __clzll((long long)some);
        if (lane == of) {
          float at = acc + (upto - m);
          int pick = -1;
#pragma unroll
          for (int j = 0; j < 8; j++) {
            at += e[j];
            if (e[j] > 0.f) last = 8 * i + j;
            if (pick < 0 && e[j] > 0.f && goal < at) pick = 8 * i + j;
          }
          if (found && pick >= 0) last = pick;
        }
        last = __shfl(last, of);
      }
      acc += __shfl(upto, 63);
    }
    const int t = 8 * nvec + s.owner;
    if (!found && t < V && __expf(ldf(p + t) * invT - M) > 0.f) last = t;
    if (lane == 0) s.found = last;
  }
  __syncthreads();
  int pick = s.found;
  if (pick < 0) {                   // no masses, or not-a-numbers among them
    float best;
    pick = row_argmax<OWNERS>(p, V, best, s.red, s.index);
  }
  if (tid == 0) {
    *out = pick;
    if (out_lp) *out_lp = ldf(p + pick) * invT - (M + __logf(total));
  }
}

// Chunks of ALL_VECS vectors a thread, `per` of them to a workgroup.  ONE: the whole row, whose
// category is chosen at once; else tops [B, slices] and masses [B, slices, OWNERS, ALL_VECS].
// Every vector of a chunk has a sum of its own, and sums, scans and walk have the order of
// sample_topp_kernel: of 151936 categories at T = 1 a border lies every 7e-6 of the mass, and
// 32-bit sums choose another of two neighbours than 64-bit ones 4 times in 1000, there and here,
// 6 times with sums in one chain.
template <typename LT, bool ONE>
__global__ __launch_bounds__(OWNERS)
void sample_all_kernel(const LT* __restrict__ logits, long* __restrict__ out,
                       float* __restrict__ out_lp, float* __restrict__ tops,
                       float* __restrict__ masses, int V, int chunks, int per, int slices,
                       float invT,
                       unsigned long long seed, unsigned long long step_imm,
                       const long* __restrict__ step_ptr) {
  __shared__ PickScratch s;
  const long row = blockIdx.x / slices;
  const int slice = blockIdx.x % slices, tid = threadIdx.x, nvec = V / 8;
  const LT* p = logits + row * (long)V;
  const int c1 = min(chunks, (slice + 1) * per);
  static_assert(ALL_VECS * OWNERS == SBLOCK, "a thread's vectors there");
  float top = -INFINITY;                   // this thread's
  f32x4 sum{0.f, 0.f, 0.f, 0.f};
  auto grow = [&](float most) {            // the exponent's subtrahend from here on
    const float now = fmaxf(top, most);
    if (now > top) sum *= __expf((top - now) * invT);
    top = now;
    return now == -INFINITY ? 0.f : now * invT;
  };
  for (int c = slice * per; c < c1; c++) {
    const int at = c * ALL_VECS * OWNERS + tid;
    Vec8<LT> v[ALL_VECS];
#pragma unroll
    for (int k = 0; k < ALL_VECS; k++) load8(p + 8L * min(at + OWNERS * k, nvec - 1), v[k]);
    float most = -INFINITY;
#pragma unroll
    for (int k = 0; k < ALL_VECS; k++) {
      if (at + OWNERS * k >= nvec) fill8(v[k]);
      float x[8];
      get8(v[k], x);
      most = fmaxf(most, max8(x));
    }
    const float M = grow(most);
    const auto add = [&](auto e) {
#pragma unroll
      for (int k = 0; k < ALL_VECS; k++) {
        float x[8];
        get8(v[k], x);
#pragma unroll
        for (int j = 0; j < 8; j++) sum[k] += e(x[j]);
      }
    };
    if (far_below(top, invT)) add([&](float l) { return __expf((l - top) * invT); });
    else add([&](float l) { return __expf(l * invT - M); });
  }
  // the last elements belong to the first owners, behind their vectors
  if (c1 == chunks && 8 * nvec + tid < V) {
    const float x = ldf(p + 8 * nvec + tid);
    const float M = grow(x);
    sum[0] += __expf(far_below(top, invT) ? (x - top) * invT : x * invT - M);
  }
  const float best = block_max<OWNERS>(top, s.red);
  if (best != -INFINITY) sum *= __expf((top - best) * invT);
  if constexpr (ONE) {
    const unsigned long long step = step_imm + (step_ptr ? (unsigned long long)*step_ptr : 0);
    __syncthreads();
    pick_of_all(s, p, V, invT, best, ((sum[0] + sum[1]) + sum[2]) + sum[3],
                hash_uniform(seed, step, (unsigned long long)row), out + row, out_lp ? out_lp + row : nullptr);
  } else {
    const long part = blockIdx.x;
    if (tid == 0) tops[part] = best;
    reinterpret_cast<f32x4*>(masses)[part * OWNERS + tid] = sum;
  }
}

template <typename LT>
__global__ __launch_bounds__(OWNERS)
void sample_all_pick_kernel(const LT* __restrict__ logits, long* __restrict__ out,
                            float* __restrict__ out_lp, const float* __restrict__ tops,
                            const float* __restrict__ masses, int V, int slices, float invT,
                            unsigned long long seed, unsigned long long step_imm,
                            const long* __restrict__ step_ptr) {
  __shared__ PickScratch s;
  const long row = blockIdx.x;
  const unsigned long long step = step_imm + (step_ptr ? (unsigned long long)*step_ptr : 0);
  float best = -INFINITY;
  f32x4 sum{0.f, 0.f, 0.f, 0.f};
  for (int i = 0; i < slices; i++) best = fmaxf(best, tops[row * slices + i]);
#pragma unroll 4
  for (int i = 0; i < slices; i++)
    sum += reinterpret_cast<const f32x4*>(masses)[(row * slices + i) * OWNERS + threadIdx.x] *
           __expf((tops[row * slices + i] - best) * invT);
  pick_of_all(s, logits + row * (long)V, V, invT, best, ((sum[0] + sum[1]) + sum[2]) + sum[3],
              hash_uniform(seed, step, (unsigned long long)row), out + row,
              out_lp ? out_lp + row : nullptr);
}

// Vectors per thread that are held in registers; 1024 threads have 128 each, so
// 19 of bf16 (155648 logits) and 8 of float32 (65536) fit beside the rest.
//
// What bounds a row: the histogram's read-add-write chains and the exponentials,
// on one CU.  151936 bf16 logits at T = 0.7, top-p 0.95, us: 8 rows 29 (with 256
// threads, five passes over memory and histograms in registers 215), 256 rows 56
// (325), 2048 rows 299 (1608); LDS float atomics in place of the private
// columns' plain adds took 221 for 8 rows.  With each vector's maximum kept, so that the
// passes after the histogram unpack only the few that matter, 8 rows 27.8 (31.0 in the same
// process), 256 rows 37.5 (40.4); four elements' histogram entries read before the first is
// written 30.5 for 8 rows: the passes are bound by the VALU of one CU.
static void launch_sampler(const torch::Tensor& logits, torch::Tensor& out, float* lp,
                           double temperature, double top_p, long seed, long step,
                           const long* step_ptr) {
  const long B = logits.size(0);
  const int V = logits.size(1), n = (V / 8 + SBLOCK - 1) / SBLOCK;
  auto stream = at::hip::getCurrentHIPStream();
  const bool half = logits.scalar_type() == torch::kBFloat16;
  if ((float)temperature == 0.f) {
    // 512 threads: 8 rows of 151936 float32 logits 10.7 us (with 1024 12.2, with 256 18.8),
    // 1024 rows of 128100 98 (106, 100); short rows are waves to start: 1024 of 1000 4.4 us
    // with 256, 6.5 with 512
#define GREEDY(LT, BLOCK)                                                                       \
  hipLaunchKernelGGL((sample_greedy_kernel<LT, BLOCK>), dim3(B), dim3(BLOCK), 0, stream,        \
                     (const LT*)logits.data_ptr(), out.data_ptr<long>(), lp, V)
    if (half) { if (V <= 8192) GREEDY(short, 256); else GREEDY(short, 512); }
    else { if (V <= 8192) GREEDY(float, 256); else GREEDY(float, 512); }
#undef GREEDY
    HIP_CHECK_LAST();
    return;
  }
  if (top_p >= 1.) {
    const int chunks = (V / 8 + ALL_VECS * OWNERS - 1) / (ALL_VECS * OWNERS);
    const int want = std::max(1L, std::min<long>(chunks, (2047 + B) / B));
    const int per = std::max(1, (chunks + want - 1) / want);
    const int slices = std::max(1, (chunks + per - 1) / per);
    const float invT = temperature > 0. ? 1.f / (float)temperature : 1.f;
    TORCH_CHECK(B * slices < 1L << 31, "sampling: too many rows");
    torch::Tensor work;
    float *tops = nullptr, *masses = nullptr;
    if (slices > 1) {
      work = torch::empty({B * slices * (SBLOCK + 1)}, logits.options().dtype(torch::kFloat32));
      masses = work.data_ptr<float>();
      tops = masses + B * slices * SBLOCK;
    }
#define LAUNCH(LT, ONE)                                                                       \
  hipLaunchKernelGGL((sample_all_kernel<LT, ONE>), dim3(B * slices), dim3(OWNERS), 0, stream, \
                     (const LT*)logits.data_ptr(), out.data_ptr<long>(), lp, tops, masses, V, \
                     chunks, per, slices, invT, (unsigned long long)seed,                     \
                     (unsigned long long)step, step_ptr)
#define PICK(LT)                                                                              \
  hipLaunchKernelGGL((sample_all_pick_kernel<LT>), dim3(B), dim3(OWNERS), 0, stream,          \
                     (const LT*)logits.data_ptr(), out.data_ptr<long>(), lp, tops, masses, V, \
                     slices, invT, (unsigned long long)seed, (unsigned long long)step, step_ptr)
    if (slices == 1) {
      if (half) LAUNCH(short, true); else LAUNCH(float, true);
    } else if (half) {
      LAUNCH(short, false);
      PICK(short);
    } else {
      LAUNCH(float, false);
      PICK(float);
    }
#undef PICK
#undef LAUNCH
    HIP_CHECK_LAST();
    return;
  }
  // A CU that has a row to itself takes the time of its VALU and LDS over the whole row: few
  // rows are divided for the first half of it.  A nucleus of few elements, as a language
  // model's, then is a few us; of rows that are flat (normal logits of deviation 1) every
  // element has to be put into a bin all the same.  Taken where neither is slower.  us, top-p 0.95,
  // one kernel / divided, logits of a language model at T = 0.7, at T = 1, where the nucleus has a
  // thousand elements | flat ones:
  //   bf16     151936   1 row  25.1 / 10.7, 37.5 / 28.9 | 43.8 / 38.3
  //                     64     28.1 / 15.1, 39.9 / 36.8 | 45.1 / 44.8
  //            128100   32     24.0 / 12.0, 34.3 / 32.6 | 38.2 / 35.5
  //                     64     25.4 / 13.7, 33.8 / 35.1 | 38.4 / 39.0   not divided
  //            107000   32     24.6 / 11.6, 33.1 / 30.7 | 35.7 / 34.9
  //             98312   32     24.3 / 11.6, 32.2 / 30.0 | 34.5 / 35.2   not divided
  //   32 bits  151936   64     48.5 / 18.9, 52.4 / 42.9 | 58.2 / 49.1
  //                     512     173 / 92,    170 / 140  |  172 / 166
  //            107000   16     26.7 / 13.0, 34.2 / 30.1 | 37.4 / 37.1
  //                     32     30.3 / 13.3, 34.9 / 33.5 | 37.5 / 38.5   not divided
  const long most = half ? (n >= 19 ? 64 : 32) : (n >= 16 ? 512 : 16);
  if (n >= 14 && n <= 20 && B <= most) {
    const int slices = (V / 8 + SLICE - 1) / SLICE;
    const int run = n <= 16 ? 32 : 40;          // half of an owner's vectors, n * 4
    const long ahead = (B * slices * 8 + 63) / 64 * 64;
    auto work = torch::empty({ahead + B * RBLOCK * run * (half ? 2 : 4)},
                             logits.options().dtype(torch::kByte));
    auto* part = (float2*)work.data_ptr();
    void* runs = (char*)work.data_ptr() + ahead;
    const float invT = temperature > 0. ? 1.f / (float)temperature : 1.f;
#define LAUNCH(LT, RUN)                                                                       \
  do {                                                                                       \
    hipLaunchKernelGGL((sample_slices_kernel<LT, RUN>), dim3(slices, B), dim3(OWNERS), 0,    \
                       stream, (const LT*)logits.data_ptr(), part, (LT*)runs, V, invT);      \
    hipLaunchKernelGGL((sample_row_kernel<LT, RUN>), dim3(B), dim3(RBLOCK), 0, stream,       \
                       (const LT*)logits.data_ptr(), out.data_ptr<long>(), lp, V, invT,      \
                       (float)top_p, (unsigned long long)seed, (unsigned long long)step,     \
                       step_ptr, part, (const LT*)runs, slices);                             \
  } while (0)
    if (half && run == 32) LAUNCH(short, 32);
    else if (half) LAUNCH(short, 40);
    else if (run == 32) LAUNCH(float, 32);
    else LAUNCH(float, 40);
#undef LAUNCH
    HIP_CHECK_LAST();
    return;
  }
#define LAUNCH(LT, NV)                                                                       \
  hipLaunchKernelGGL((sample_topp_kernel<LT, NV>), dim3(B), dim3(SBLOCK), 0, stream,         \
                     (const LT*)logits.data_ptr(), out.data_ptr<long>(), lp, V,              \
                     (float)temperature, (float)top_p, (unsigned long long)seed,             \
                     (unsigned long long)step, step_ptr)
  if (half) {
    if (n <= 4) LAUNCH(short, 4);
    else if (n <= 16) LAUNCH(short, 16);
    else if (n <= 19) LAUNCH(short, 19);
    else LAUNCH(short, 0);
  } else {
    if (n <= 8) LAUNCH(float, 8);
    else LAUNCH(float, 0);
  }
#undef LAUNCH
  HIP_CHECK_LAST();
}

torch::Tensor sample_topp(torch::Tensor logits, double temperature, double top_p,
                          long seed, long step) {
  TORCH_CHECK(logits.dim() == 2 && logits.is_contiguous());
  const bool half = logits.scalar_type() == torch::kBFloat16;
  TORCH_CHECK(half || logits.scalar_type() == torch::kFloat32, "logits must be bf16 or float32");
  const long B = logits.size(0);
  auto out = torch::empty({B}, logits.options().dtype(torch::kLong));
  if (B == 0) return out;
  launch_sampler(logits, out, nullptr, temperature, top_p, seed, step, nullptr);
  return out;
}

std::vector<torch::Tensor> sample_topp_dev(torch::Tensor logits, double temperature,
                                           double top_p, long seed, torch::Tensor step,
                                           long ahead) {
  // step: int64 [1] device tensor, read inside the kernel, and `ahead` more — safe under
  // hipGraph capture/replay (the immediate-arg form would freeze the step).
  // Also returns the chosen token's logprob (vLLM logprobs parity).
  TORCH_CHECK(logits.dim() == 2 && logits.is_contiguous());
  const bool half = logits.scalar_type() == torch::kBFloat16;
  TORCH_CHECK(half || logits.scalar_type() == torch::kFloat32, "logits must be bf16 or float32");
  TORCH_CHECK(step.scalar_type() == torch::kLong && step.is_cuda());
  const long B = logits.size(0);
  auto out = torch::empty({B}, logits.options().dtype(torch::kLong));
  auto lp = torch::empty({B}, logits.options().dtype(torch::kFloat32));
  if (B == 0) return {out, lp};
  launch_sampler(logits, out, lp.data_ptr<float>(), temperature, top_p, seed, ahead,
                 step.data_ptr<long>());
  return {out, lp};
}

// ------------------------------------------------------------ decode batch
// What a decode step does to its rows beside the model: where each row's token
// goes in the cache, and afterwards what the sampled token changes, the counter of the
// sampling among it.  A thread a
// row; bound by the launch, of which tensor operations took 26 a step: a rollout
// of 64 rows and 96 tokens through 6 layers went from 85.2 to 78.5 ms.
__global__ __launch_bounds__(256)
void decode_inputs_kernel(const int* __restrict__ lens, const int* __restrict__ bt,
                          long* __restrict__ pos, long* __restrict__ slots, int B, int P, int ps) {
  const int b = blockIdx.x * 256 + threadIdx.x;
  if (b >= B) return;
  const int at = lens[b] - 1;
  pos[b] = at;
  slots[b] = (long)bt[(long)b * P + min(max(at, 0) / ps, P - 1)] * ps + max(at, 0) % ps;
}

__global__ __launch_bounds__(256)
void decode_commit_kernel(const long* __restrict__ tokens, const float* __restrict__ lps,
                          long* __restrict__ out, float* __restrict__ lp, int* __restrict__ count,
                          int* __restrict__ lens, long* __restrict__ last,
                          bool* __restrict__ finished, int B, int most, long stop,
                          bool has_stop, long* __restrict__ step) {
  const int b = blockIdx.x * 256 + threadIdx.x;
  if (b == 0 && step) *step += 1;
  if (b >= B) return;
  const int n = count[b];
  if (finished[b] || n >= most) {
    finished[b] = finished[b] || n >= most;
    return;
  }
  const long tok = tokens[b];
  out[(long)b * most + n] = tok;
  if (lps) lp[(long)b * most + n] = lps[b];
  count[b] = n + 1;
  lens[b]++;
  last[b] = tok;
  finished[b] = (has_stop && tok == stop) || n + 1 >= most;
}

std::vector<torch::Tensor> decode_inputs(torch::Tensor lens, torch::Tensor bt, long page_size) {
  const int B = lens.size(0);
  TORCH_CHECK(lens.is_cuda() && bt.is_cuda() && bt.dim() == 2 && bt.size(0) == B &&
              bt.size(1) > 0 && page_size > 0, "decode_inputs: lengths [B], pages [B, P]");
  TORCH_CHECK(lens.scalar_type() == at::kInt && bt.scalar_type() == at::kInt &&
              lens.is_contiguous() && bt.is_contiguous(), "decode_inputs: contiguous int32");
  auto pos = torch::empty({B}, lens.options().dtype(at::kLong)), slots = torch::empty_like(pos);
  if (B)
    hipLaunchKernelGGL(decode_inputs_kernel, dim3((B + 255) / 256), dim3(256), 0,
                       c10::hip::getCurrentHIPStream(), lens.data_ptr<int>(), bt.data_ptr<int>(),
                       pos.data_ptr<long>(), slots.data_ptr<long>(), B, (int)bt.size(1),
                       (int)page_size);
  HIP_CHECK_LAST();
  return {pos, slots};
}

void decode_commit(torch::Tensor tokens, c10::optional<torch::Tensor> lps, torch::Tensor out,
                   torch::Tensor lp, torch::Tensor count, torch::Tensor lens, torch::Tensor last,
                   torch::Tensor finished, c10::optional<long> stop,
                   c10::optional<torch::Tensor> step) {
  const int B = out.size(0), most = out.size(1);
  TORCH_CHECK(!step || (step->is_cuda() && step->scalar_type() == at::kLong && step->numel() == 1),
              "decode_commit: an int64 step");
  for (const auto& t : {tokens, count, lens, last, finished})
    TORCH_CHECK(t.is_cuda() && t.is_contiguous() && t.dim() == 1 && t.size(0) == B,
                "decode_commit: one contiguous entry a row");
  TORCH_CHECK(out.is_contiguous() && lp.is_contiguous() && lp.sizes() == out.sizes() &&
              out.scalar_type() == at::kLong && lp.scalar_type() == at::kFloat &&
              tokens.scalar_type() == at::kLong && last.scalar_type() == at::kLong &&
              count.scalar_type() == at::kInt && lens.scalar_type() == at::kInt &&
              finished.scalar_type() == at::kBool, "decode_commit: types");
  TORCH_CHECK(!lps || (lps->is_cuda() && lps->is_contiguous() && lps->numel() == B &&
                       lps->scalar_type() == at::kFloat), "decode_commit: log-probabilities");
  if (B)
    hipLaunchKernelGGL(decode_commit_kernel, dim3((B + 255) / 256), dim3(256), 0,
                       c10::hip::getCurrentHIPStream(), tokens.data_ptr<long>(),
                       lps ? lps->data_ptr<float>() : nullptr, out.data_ptr<long>(),
                       lp.data_ptr<float>(), count.data_ptr<int>(), lens.data_ptr<int>(),
                       last.data_ptr<long>(), finished.data_ptr<bool>(), B, most,
                       stop.value_or(0), stop.has_value(),
                       step ? step->data_ptr<long>() : nullptr);
  HIP_CHECK_LAST();
}
