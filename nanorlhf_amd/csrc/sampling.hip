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
#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>

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
