// Latent attention over the paged cache of normed latents c [P, 16, R]: every
// head's key and value are linear in c.  Queries arrive multiplied by their
// head's key map (qa, R wide), so a score is qa . c, and what leaves is the
// softmax-weighted sum of c, which the caller passes through the value maps.
//
// latent_attn (bf16, MFMA): one workgroup of 4 waves per (sequence, 16 rows, part
// of the context); a row is a (token, head) pair, tokens outermost.  Every wave
// walks pages of its own (16 tokens, contiguous in memory) with a running maximum
// and sum of its own and shares nothing with the others until the end: pages come
// to its part of LDS by direct loads, up to three ahead, S^T = C Q^T reads them
// along the latent and O^T += C^T P^T turned around (ds_read_tr16_b64).  Scores of
// one row lie in one lane's column, and as they come out of the first product
// they are the second's operand.  latent_merge joins parts of a split context.
//
// latent_attn_plain: one wave per (token, head), scalar products in 32-bit.
#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>

#include <type_traits>

#include "common.h"
#include "checks.h"

// ---------------------------------------------- norm and write the latents
// One wave per row: c / sqrt(mean(c^2) + eps) * w, zeros in the pad columns.
// VEC neighbouring elements per lane; the first 64 VEC stay in registers.
template <typename T, int VEC>
__global__ __launch_bounds__(256) void latent_append_kernel(
    const T* __restrict__ c, long ldc, const T* __restrict__ w, const long* __restrict__ slots,
    T* __restrict__ cache, long rows, int R, int RP, float eps) {
  const int lane = threadIdx.x & 63;
  const long row = blockIdx.x * 4L + (threadIdx.x >> 6);
  if (row >= rows) return;
  const T* src = c + row * ldc;
  T* dst = cache + slots[row] * (long)RP;
  const int e0 = lane * VEC;
  float x[VEC] = {}, g[VEC] = {};
  if (e0 < R) {
    ldv<VEC>(src + e0, x);
    ldv<VEC>(w + e0, g);
  }
  float ss = 0.f;
#pragma unroll
  for (int j = 0; j < VEC; j++) ss += x[j] * x[j];
  for (int e = e0 + 64 * VEC; e < R; e += 64 * VEC) {
    float y[VEC];
    ldv<VEC>(src + e, y);
#pragma unroll
    for (int j = 0; j < VEC; j++) ss += y[j] * y[j];
  }
  const float inv = 1.f / sqrtf(wave_sum(ss) / (float)R + eps);
  auto put = [&](int e) {                    // x and g are zero past R
#pragma unroll
    for (int j = 0; j < VEC; j++) x[j] = x[j] * inv * g[j];
    stv<VEC>(dst + e, x);
  };
  if (e0 < RP) put(e0);
  for (int e = e0 + 64 * VEC; e < RP; e += 64 * VEC) {
    if (e < R) {
      ldv<VEC>(src + e, x);
      ldv<VEC>(w + e, g);
    } else {
#pragma unroll
      for (int j = 0; j < VEC; j++) x[j] = 0.f;
    }
    put(e);
  }
}

// ---------------------------------------------------- the matrix-core kernel
struct LatentArgs {
  const short* qa;       // [T, H, RP]
  const short* cache;    // [P, 16, RP]
  const int* cu;         // [B + 1] first token of each sequence, or null: one each
  const int* seq_lens;   // [B] keys, the step's own included
  const int* bt;         // [B, maxP]
  short* out;            // [T, H, RP], if not split
  float* part;           // [units, splits, 16, RP] sums, and after them
  float* ms;             // [units, splits, 16, 2] maximum (log2) and weight
  int H, maxP, splits;
  float scale;
  int B, budget;         // one token each: workgroups to divide all pages among, or 0
  int2* plan;            // [B] a sequence's first workgroup, and how many it has
};

// Which part of which sequence workgroup w of a.budget has: every sequence is divided into as
// many parts of at most `per` pages as it takes, `per` being about the least (to a sixteenth)
// with which all parts are at most the budget.  A wave's lane looks at four sequences; all waves
// come to the same.
struct LatentPart { int seq, z, per, parts, length; };
DEVINL bool latent_part(const LatentArgs& a, int w, LatentPart& out) {
  const int lane = threadIdx.x & 63;
  int lens[4], pages[4];
  float sum = 0.f, longest = 0.f;
#pragma unroll
  for (int i = 0; i < 4; i++) lens[i] = a.seq_lens[min(4 * lane + i, a.B - 1)];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    asm volatile("" : "+v"(lens[i]));        // asked for together
    pages[i] = 4 * lane + i < a.B ? max((lens[i] - 1) / 16 + 1, 1) : 0;
  }
#pragma unroll
  for (int i = 0; i < 4; i++) {
    sum += (float)pages[i];
    longest = fmaxf(longest, (float)pages[i]);
  }
  const float total = wave_sum(sum);
  const int most = (int)wave_max(longest);
  auto parts = [&](int n, int per, float inv) {      // n / per, rounded up
    int q = (int)((float)(n + per - 1) * inv);
    if (q * per > n + per - 1) q--;
    if ((q + 1) * per <= n + per - 1) q++;
    return q;
  };
  // two pages to a wave at least, and what the merge's lanes can hold
  int low = max(max(8, (most + 63) / 64), (int)(total / (float)a.budget));
  int per = max(low, min(most, (int)(total / (float)(a.budget - a.B)) + 1));
  while (per - low > low / 16) {
    const int mid = (low + per) / 2;
    const float inv = 1.f / (float)mid;
    float n = 0.f;
#pragma unroll
    for (int i = 0; i < 4; i++) n += (float)parts(pages[i], mid, inv);
    if (wave_sum(n) <= (float)a.budget) per = mid;
    else low = mid + 1;
  }
  int c[4], mine = 0;
#pragma unroll
  for (int i = 0; i < 4; i++) {
    c[i] = parts(pages[i], per, 1.f / (float)per);
    mine += c[i];
  }
  int upto = mine;           // sums over the lanes before: row_shr:1, 2, 4, 8, then the rows'
  auto shift = [&](auto ctrl) {
    upto += __builtin_amdgcn_update_dpp(0, upto, decltype(ctrl)::value, 0xf, 0xf, true);
  };
  shift(std::integral_constant<int, 0x111>{});
  shift(std::integral_constant<int, 0x112>{});
  shift(std::integral_constant<int, 0x114>{});
  shift(std::integral_constant<int, 0x118>{});
  {
    const int r0 = __builtin_amdgcn_readlane(upto, 15), r1 = r0 + __builtin_amdgcn_readlane(upto, 31);
    const int r2 = r1 + __builtin_amdgcn_readlane(upto, 47), r = lane >> 4;
    upto += r == 0 ? 0 : r == 1 ? r0 : r == 2 ? r1 : r2;
  }
  const unsigned long long hit = __ballot(w >= upto - mine && w < upto);
  if (!hit) return false;
  const int at = __ffsll(hit) - 1;
  int z = w - __builtin_amdgcn_readlane(upto - mine, at), seq = 4 * at, n = 0, length = 0;
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const int here = __builtin_amdgcn_readlane(c[i], at);
    if (n == 0 && z < here) {
      n = here;
      seq = 4 * at + i;
      length = __builtin_amdgcn_readlane(lens[i], at);
    } else if (n == 0) {
      z -= here;
    }
  }
  out = {seq, z, per, n, length};
  return true;
}

// A page's 16-byte chunks are exchanged (xor) by row, so that 16 rows at one
// column (scores) and 4 rows at 4 columns (turned around) meet all banks.
template <int RP>
DEVINL int page_swz(int row) {
  if constexpr (RP == 64)        // two rows per 256 bytes
    return ((row >> 1) & 1) << 1 | ((row >> 2) & 1) << 2 | (row >> 3);
  else
    return (row & 3) << 2 | ((row >> 2) & 1) << 1 | (row >> 3);
}

// What bounds it: reading the latents, and their uneven lengths.  128 contexts of
// about 2000 latents of 512, 12 heads: 63 us (4.2 TB/s) with two parts each, one
// workgroup per CU; with whole tiles of 64 tokens going through registers and
// four barriers per tile it took 116.  Before fragments were read ahead (72 us) four
// parts took 9 us more than two (a part's first loads and sums), two waves per
// workgroup 2 more.
template <int RP, bool ALL>
__global__ __launch_bounds__(256) void latent_attn_kernel(LatentArgs a) {
  constexpr int NW = 4, NC = RP / 32, NT = RP / 16, CH = RP / 8;
  constexpr int PAGE = 16 * RP;                          // elements
  constexpr int LOADS = PAGE / 512;                      // direct loads per page
  constexpr int NBUF = RP >= 512 ? 2 : 4;
  // pages of each wave; at the end its sums, 16 x RP floats
  __shared__ __attribute__((aligned(1024))) short buf[NW][NBUF * PAGE];
  __shared__ float Lm[NW][16], Ls[NW][16];
  int seq = blockIdx.y, z = blockIdx.z, splits = a.splits, per = 0, length = 0;
  if constexpr (ALL) {
    LatentPart mine;
    if (!latent_part(a, blockIdx.y, mine)) return;
    seq = mine.seq;
    z = mine.z;
    splits = mine.parts;
    per = mine.per;
    length = mine.length;
    if (z == 0 && blockIdx.x == 0 && threadIdx.x == 0) a.plan[seq] = int2{(int)blockIdx.y, splits};
  }
  const int t0 = !ALL && a.cu ? a.cu[seq] : seq;
  const int nq = !ALL && a.cu ? a.cu[seq + 1] - t0 : 1;
  const int R = nq * a.H, r0 = blockIdx.x * 16;
  if (r0 >= R) return;
  const int start = (ALL ? length : a.seq_lens[seq]) - nq;
  const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lo = lane & 15, hi = lane >> 4;
  const int row = min(r0 + lo, R - 1);
  const int qpos = start + row / a.H;         // of this lane's row
  const int npages = (start + min(r0 + 15, R - 1) / a.H) / 16 + 1;
  if (!ALL) per = (npages + splits - 1) / splits;
  const int p0 = z * per, p1 = min(npages, p0 + per);
  // scalar loads: a vector load would be waited for behind the pages under way
  typedef const __attribute__((address_space(4))) int* const_ints;
  const const_ints btb = (const_ints)(size_t)(a.bt + (long)seq * a.maxP);

  auto fetch = [&](int page, int slot) {
    const short* src = a.cache + (long)btb[page] * PAGE;
#pragma unroll
    for (int j = 0; j < LOADS; j++) {
      const int idx = 64 * j + lane, r = idx / CH, c = (idx % CH) ^ page_swz<RP>(r);
      load_to_lds16(src, (r * CH + c) * 16, &buf[wid][slot * PAGE + 512 * j]);
    }
  };
  int ahead = p0 + wid;
#pragma unroll
  for (int b = 0; b < NBUF; b++, ahead += NW)
    if (ahead < p1) fetch(ahead, b);

  bf16x8l qf[NC];
#pragma unroll
  for (int q = 0; q < NC; q++)
    qf[q] = frag(a.qa + ((long)t0 * a.H + row) * RP + 32 * q + 8 * hi);
  // waited for here, once: in the loop the wait would take the pages' loads along
#pragma unroll
  for (int q = 0; q < NC; q++) asm volatile("" : "+v"(qf[q]));

  // this lane's part of a page, by rows (scores) and turned around
  typedef __attribute__((address_space(3))) char* lds_bytes;
  typedef __attribute__((address_space(3))) const bf16x8l* lds_frag;
  typedef __attribute__((address_space(3))) s16x4* lds_s16x4;
  const int tr = 4 * hi + (lo >> 2);
  const unsigned buf0 = lds_address(buf[wid]);
  const unsigned row_at = lo * 2 * RP + ((hi ^ page_swz<RP>(lo)) << 4);
  const unsigned col_at = tr * 2 * RP + ((((lo & 3) >> 1) ^ page_swz<RP>(tr)) << 4) + (lo & 1) * 8;

  float m = -INFINITY, sum = 0.f;             // of row lo
  f32x4 acc[NT];                              // O^T: latent columns 16 t + 4 hi + r, row lo
#pragma unroll
  for (int t = 0; t < NT; t++) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  const float sl2 = a.scale * 1.4426950408889634f;
  int slot = 0;
  for (int pg = p0 + wid; pg < p1; pg += NW) {
    // pages behind this one that are on their way
    if (pg + NW * (NBUF - 1) < p1) wait_loads<LOADS * (NBUF - 1)>();
    else wait_loads<0>();
    // Another fragment along the latent is an xor of its chunk, which has the bits below
    // 256 bytes to itself, and an offset.  At 512 that makes a few addresses; one for each
    // fragment would leave no registers to read ahead of the products (1 x 200 tokens
    // of 12 heads 14.2 us, 15.5).  Narrower latents have them: 128 x 2000 of 256 38 us, 39.5.
    const unsigned page = buf0 + slot * (PAGE * 2), ra = page + row_at, ca = page + col_at;
    const short* C = &buf[wid][slot * PAGE];
    auto by_row = [&](int q) {
      if constexpr (RP >= 512) return *(lds_frag)((lds_bytes)(ra ^ (q & 3) << 6) + (q >> 2) * 256);
      else return frag(C + lo * RP + (((4 * q + hi) ^ page_swz<RP>(lo)) << 3));
    };
    auto turned = [&](int t) {
      if constexpr (RP >= 512)
        return (lds_s16x4)((lds_bytes)(ca ^ (t & 7) << 5) + (t >> 3) * 256);
      else
        return (lds_s16x4)(C + tr * RP + (((2 * t + ((lo & 3) >> 1)) ^ page_swz<RP>(tr)) << 3) +
                           (lo & 1) * 4);
    };
    f32x4 s2[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int q = 0; q < NC; q++)
      s2[q & 1] = mfma16l(by_row(q), qf[q], s2[q & 1]);
    float x[4], top = -INFINITY;
#pragma unroll
    for (int r = 0; r < 4; r++) {
      x[r] = 16 * pg + 4 * hi + r > qpos ? -INFINITY : (s2[0][r] + s2[1][r]) * sl2;
      top = fmaxf(top, x[r]);
    }
    top = fmaxf(top, __shfl_xor(top, 16));
    top = fmaxf(top, __shfl_xor(top, 32));
    float alpha = 1.f;
    // a row's largest weight is 1 exactly, so that it is not rounded
    if (__any(!(top <= m))) {
      const float mn = fmaxf(m, top);
      alpha = m == -INFINITY ? 0.f : exp2f(m - mn);
      m = mn;
#pragma unroll
      for (int t = 0; t < NT; t++) acc[t] *= alpha;
    }
    const float mm = m == -INFINITY ? 0.f : m;
    s16x4 pf;
    float rs = 0.f;
#pragma unroll
    for (int r = 0; r < 4; r++) {
      pf[r] = f2bf(exp2f(x[r] - mm));         // normed by the sum of the weights as rounded
      rs += bf2f(pf[r]);
    }
    rs += __shfl_xor(rs, 16);
    rs += __shfl_xor(rs, 32);
    sum = sum * alpha + rs;
#pragma unroll
    for (int t = 0; t < NT; t++)
      acc[t] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(
          __builtin_amdgcn_ds_read_tr16_b64_v4i16(turned(t)), pf, acc[t], 0, 0, 0);
    if (ahead < p1) {
      lds_fence_wave_kv();                    // this page's reads are done
      fetch(ahead, slot);
      ahead += NW;
    }
    slot = slot + 1 == NBUF ? 0 : slot + 1;
  }

  // ---- the four waves' sums, in their own LDS (chunks of 4 exchanged by row)
  lds_fence_wave_kv();
  float* own = reinterpret_cast<float*>(buf[wid]);
#pragma unroll
  for (int t = 0; t < NT; t++)
    *reinterpret_cast<f32x4*>(own + lo * RP + (((4 * t + hi) ^ lo) << 2)) = acc[t];
  if (hi == 0) { Lm[wid][lo] = m; Ls[wid][lo] = sum; }
  __syncthreads();
  const long unit = ALL ? (long)blockIdx.y * gridDim.x + blockIdx.x
                        : ((long)blockIdx.y * gridDim.x + blockIdx.x) * splits + z;
  // four rows to a wave; all sums ahead of the first store, so that their reads overlap
  constexpr int NK = RP / 64;
  f32x4 o[NK];
  float M[NK], S[NK];
#pragma unroll
  for (int k = 0; k < NK; k++) {
    const int i = lane + 64 * k, r = 4 * wid + i / (RP / 4), c = i % (RP / 4);
    M[k] = Lm[0][r];
#pragma unroll
    for (int w = 1; w < NW; w++) M[k] = fmaxf(M[k], Lm[w][r]);
    const float Mf = M[k] == -INFINITY ? 0.f : M[k];
    S[k] = 0.f;
    o[k] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < NW; w++) {
      const float f = exp2f(Lm[w][r] - Mf);
      S[k] += Ls[w][r] * f;
      o[k] += *reinterpret_cast<const f32x4*>(reinterpret_cast<float*>(buf[w]) + r * RP +
                                              ((c ^ r) << 2)) * f;
    }
  }
#pragma unroll
  for (int k = 0; k < NK; k++) {
    const int i = lane + 64 * k, r = 4 * wid + i / (RP / 4), c = i % (RP / 4);
    if (r0 + r >= R) continue;
    if (splits > 1) {
      *reinterpret_cast<f32x4*>(a.part + (unit * 16 + r) * RP + 4 * c) = o[k];
      if (c == 0) {
        a.ms[(unit * 16 + r) * 2] = M[k];
        a.ms[(unit * 16 + r) * 2 + 1] = S[k];
      }
    } else {
      const float inv = 1.f / S[k];
      const float y[4] = {o[k][0] * inv, o[k][1] * inv, o[k][2] * inv, o[k][3] * inv};
      stv<4>(a.out + ((long)t0 * a.H + r0 + r) * RP + 4 * c, y);
    }
  }
}

// One workgroup per (16-row unit, row): the parts of a split context joined.  A chain of
// latencies, so up to MOST parts are asked for at once with their shares.
template <int MOST, bool ALL>
__global__ __launch_bounds__(128) void latent_merge_kernel(LatentArgs a, int RP, int units_x) {
  const int unit = blockIdx.x, rr = blockIdx.y;
  const int seq = unit / units_x, r0 = unit % units_x * 16;
  const int z = threadIdx.x & 63;
  int splits = a.splits, step = 1;
  long first = (long)unit * splits;                    // of parts
  if constexpr (ALL) {
    const int2 has = a.plan[seq];
    splits = has.y;
    if (splits < 2) return;                            // written as it is
    first = (long)has.x * units_x + unit % units_x;
    step = units_x;
  }
  const float* ms = a.ms + (first * 16 + rr) * 2;
  const float* p = a.part + (first * 16 + rr) * RP;
  const float2 w = z < splits ? *reinterpret_cast<const float2*>(ms + z * step * 32)
                              : float2{-INFINITY, 0.f};
  f32x4 x[MOST ? MOST : 1];
#pragma unroll
  for (int i = 0; i < MOST; i++)
    x[i] = *reinterpret_cast<const f32x4*>(p + (long)min(i, splits - 1) * step * 16 * RP +
                                           min((int)threadIdx.x * 4, RP - 4));
#pragma unroll
  for (int i = 0; i < MOST; i++) asm volatile("" : "+v"(x[i]));
  const int t0 = a.cu ? a.cu[seq] : seq;
  const int nq = a.cu ? a.cu[seq + 1] - t0 : 1;
  if (r0 + rr >= nq * a.H) return;
  const float f = exp2f(w.x - wave_max(w.x));
  float share = f / wave_sum(w.y * f);
  asm volatile("" : "+v"(share));         // of every lane, those too that have no column below
  // Part i's share of the result.  Of many parts through LDS: 16 x 8000 latents, in 16 parts, took
  // 48.5 us so and 51.3 with a lane read for each; 8 x 4000 of 256 by pages, in some 28, the merge
  // alone 3.9 and 12.0.
  __shared__ float shares[MOST ? 1 : 64];
  if constexpr (MOST == 0) {
    if (threadIdx.x < 64) shares[z] = share;
    __syncthreads();
  }
  auto of = [&](int i) {
    if constexpr (MOST == 0) return shares[i];
    else return __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(share), i));
  };
  short* out = a.out + ((long)t0 * a.H + r0 + rr) * RP;
  for (int d = threadIdx.x * 4; d < RP; d += 512) {
    float o[4] = {};
#pragma unroll
    for (int i = 0; i < MOST; i++)
      if (i < splits) {
        const float g = of(i);
#pragma unroll
        for (int j = 0; j < 4; j++) o[j] += g * x[i][j];
      }
#pragma unroll 4
    for (int i = MOST; i < splits; i++) {
      const float g = of(i);
      float y[4];
      ldv<4>(p + (long)i * step * 16 * RP + d, y);
#pragma unroll
      for (int j = 0; j < 4; j++) o[j] += g * y[j];
    }
    stv<4>(out + d, o);
  }
}

// Contexts one after the other, each from row first[b]; zeros behind its end.
__global__ __launch_bounds__(256) void latent_gather_kernel(
    const short* __restrict__ cache, const int* __restrict__ bt, const int* __restrict__ seq_lens,
    const int* __restrict__ first, short* __restrict__ out, long rows, int B, int maxP, int RP) {
  const int nvec = RP / 8;
  const long idx = (long)blockIdx.x * 256 + threadIdx.x;
  if (idx >= rows * nvec) return;
  const long row = idx / nvec;
  const int e = (int)(idx % nvec) * 8;
  int b = 0, end = B;                          // the last b with first[b] <= row
  while (end - b > 1) {
    const int mid = (b + end) >> 1;
    if (first[mid] <= row) b = mid; else end = mid;
  }
  const int pos = (int)(row - first[b]);
  s16x8 x{};
  if (pos < seq_lens[b])
    x = *reinterpret_cast<const s16x8*>(
        cache + ((long)bt[(long)b * maxP + (pos >> 4)] * 16 + (pos & 15)) * RP + e);
  *reinterpret_cast<s16x8*>(out + row * RP + e) = x;
}

// -------------------------------------------------------- plain, any type
template <typename T>
__global__ __launch_bounds__(256) void latent_plain_kernel(
    const T* __restrict__ qa, const T* __restrict__ cache, const int* __restrict__ row_seq,
    const long* __restrict__ positions, const int* __restrict__ bt, T* __restrict__ out,
    long rows, int H, int R, int maxP, float scale) {
  extern __shared__ float sh[];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const long unit = blockIdx.x * 4L + wid;
  if (unit >= rows * H) return;
  float *qs = sh + (long)wid * (2 * R + 64), *acc = qs + R, *ps = acc + R;
  const long t = unit / H;
  const int pos = (int)positions[t];
  const int* btb = bt + (long)row_seq[t] * maxP;
  for (int d = lane; d < R; d += 64) {
    qs[d] = ldf(qa + unit * R + d);
    acc[d] = 0.f;
  }
  lds_fence_wave_kv();
  float m = -INFINITY, sum = 0.f;
  for (int k0 = 0; k0 <= pos; k0 += 64) {
    const int ki = k0 + lane;
    float s = -INFINITY;
    if (ki <= pos) {
      const T* cr = cache + ((long)btb[min(ki >> 4, maxP - 1)] * 16 + (ki & 15)) * R;
      float dot = 0.f;
      for (int d = 0; d < R; d += 4) {
        float x[4];
        ldv<4>(cr + d, x);
#pragma unroll
        for (int j = 0; j < 4; j++) dot += x[j] * qs[d + j];
      }
      s = dot * scale;
    }
    const float mn = fmaxf(m, wave_max(s));
    const float alpha = (m == -INFINITY) ? 0.f : expf(m - mn);
    const float p = (s == -INFINITY) ? 0.f : expf(s - mn);
    m = mn;
    sum = sum * alpha + wave_sum(p);
    ps[lane] = p;
    lds_fence_wave_kv();
    const int n = min(64, pos + 1 - k0);
    for (int d = lane; d < R; d += 64) {
      float a = acc[d] * alpha;
      for (int j = 0; j < n; j++)
        a += ps[j] * ldf(cache + ((long)btb[min((k0 + j) >> 4, maxP - 1)] * 16 + ((k0 + j) & 15)) *
                                     R + d);
      acc[d] = a;
    }
    lds_fence_wave_kv();
  }
  for (int d = lane; d < R; d += 64) stf(out + unit * R + d, acc[d] / sum);
}

// ======================================================== host wrappers ==
void latent_append(torch::Tensor c, torch::Tensor w, torch::Tensor slots, torch::Tensor cache,
                   double eps) {
  const long T = c.size(0), R = c.size(1);
  on_gpu({c, w, slots, cache});
  TORCH_CHECK(c.dim() == 2 && c.stride(1) == 1 && w.is_contiguous() && w.numel() == R);
  TORCH_CHECK(cache.dim() == 3 && cache.is_contiguous() && cache.size(1) == 16 && cache.size(2) >= R);
  TORCH_CHECK(w.scalar_type() == c.scalar_type() && cache.scalar_type() == c.scalar_type());
  TORCH_CHECK(slots.scalar_type() == torch::kLong && slots.is_contiguous() && slots.numel() == T);
  if (T == 0) return;
  auto stream = at::hip::getCurrentHIPStream();
  const long es = c.element_size();
  const bool vec = R % 8 == 0 && cache.size(2) % 8 == 0 && c.stride(0) * es % 16 == 0 &&
                   (uintptr_t)c.data_ptr() % 16 == 0 && (uintptr_t)w.data_ptr() % 16 == 0;
#define LAUNCH(TT, VEC)                                                                        \
  hipLaunchKernelGGL((latent_append_kernel<TT, VEC>), dim3((T + 3) / 4), dim3(256), 0, stream, \
                     (const TT*)c.data_ptr(), (long)c.stride(0), (const TT*)w.data_ptr(),      \
                     slots.data_ptr<long>(), (TT*)cache.data_ptr(), T, (int)R,                 \
                     (int)cache.size(2), (float)eps)
  if (c.scalar_type() == torch::kBFloat16) {
    if (vec) LAUNCH(short, 8); else LAUNCH(short, 1);
  } else {
    TORCH_CHECK(c.scalar_type() == torch::kFloat32);
    if (vec) LAUNCH(float, 4); else LAUNCH(float, 1);
  }
#undef LAUNCH
  HIP_CHECK_LAST();
}

static void check_latent(const torch::Tensor& qa, const torch::Tensor& cache,
                         const torch::Tensor& bt) {
  on_gpu({qa, cache, bt});
  TORCH_CHECK(qa.dim() == 3 && qa.is_contiguous());
  TORCH_CHECK(cache.dim() == 3 && cache.is_contiguous() && cache.size(1) == 16 &&
              cache.size(2) == qa.size(2) && cache.scalar_type() == qa.scalar_type());
  TORCH_CHECK(bt.scalar_type() == torch::kInt && bt.is_contiguous() && bt.dim() == 2 && bt.size(1) > 0);
}

torch::Tensor latent_attn_plain(torch::Tensor qa, torch::Tensor cache, torch::Tensor row_seq,
                                torch::Tensor positions, torch::Tensor bt, double scale) {
  check_latent(qa, cache, bt);
  const long T = qa.size(0), H = qa.size(1), R = qa.size(2);
  on_gpu({row_seq, positions});
  TORCH_CHECK(row_seq.scalar_type() == torch::kInt && row_seq.is_contiguous() && row_seq.numel() == T);
  TORCH_CHECK(positions.scalar_type() == torch::kLong && positions.is_contiguous() && positions.numel() == T);
  const size_t lds = 4 * sizeof(float) * (2 * R + 64);
  TORCH_CHECK(R % 4 == 0 && lds <= 65536, "unsupported latent width ", R);
  auto out = torch::empty_like(qa);
  if (T == 0) return out;
  auto stream = at::hip::getCurrentHIPStream();
#define LAUNCH(TT)                                                                              \
  hipLaunchKernelGGL((latent_plain_kernel<TT>), dim3((T * H + 3) / 4), dim3(256), lds, stream,  \
                     (const TT*)qa.data_ptr(), (const TT*)cache.data_ptr(),                     \
                     row_seq.data_ptr<int>(), positions.data_ptr<long>(), bt.data_ptr<int>(),   \
                     (TT*)out.data_ptr(), T, (int)H, (int)R, (int)bt.size(1), (float)scale)
  if (qa.scalar_type() == torch::kBFloat16) LAUNCH(short);
  else {
    TORCH_CHECK(qa.scalar_type() == torch::kFloat32);
    LAUNCH(float);
  }
#undef LAUNCH
  HIP_CHECK_LAST();
  return out;
}

static void check_lens(const torch::Tensor& seq_lens, const torch::Tensor& bt) {
  TORCH_CHECK(seq_lens.is_cuda() && seq_lens.scalar_type() == torch::kInt &&
              seq_lens.is_contiguous() && bt.size(0) == seq_lens.numel());
}

// [rows, RP]: the contexts of B sequences, sequence b's from row first[b] on
// (multiples of 64, first[B] == rows)
torch::Tensor latent_gather(torch::Tensor cache, torch::Tensor bt, torch::Tensor seq_lens,
                            torch::Tensor first, long rows) {
  on_gpu({cache, bt, first});
  TORCH_CHECK(cache.dim() == 3 && cache.is_contiguous() && cache.size(1) == 16 &&
              cache.scalar_type() == torch::kBFloat16 && cache.size(2) % 8 == 0);
  TORCH_CHECK(bt.scalar_type() == torch::kInt && bt.is_contiguous() && bt.dim() == 2);
  check_lens(seq_lens, bt);
  const long B = seq_lens.numel(), RP = cache.size(2);
  TORCH_CHECK(first.scalar_type() == torch::kInt && first.is_contiguous() && first.numel() == B + 1 &&
              rows % 64 == 0);
  auto out = torch::empty({rows, RP}, cache.options());
  if (rows == 0) return out;
  const long n = rows * (RP / 8);
  hipLaunchKernelGGL(latent_gather_kernel, dim3((n + 255) / 256), dim3(256), 0,
                     at::hip::getCurrentHIPStream(), (const short*)cache.data_ptr(),
                     bt.data_ptr<int>(), seq_lens.data_ptr<int>(), first.data_ptr<int>(),
                     (short*)out.data_ptr(), rows, (int)B, (int)bt.size(1), (int)RP);
  HIP_CHECK_LAST();
  return out;
}

// qa [T, H, RP] -> [T, H, RP].  cu null: one token of each sequence; else the
// portions cu, of which the longest has max_q tokens.
torch::Tensor latent_attn(torch::Tensor qa, torch::Tensor cache, c10::optional<torch::Tensor> cu,
                          torch::Tensor seq_lens, torch::Tensor bt, long max_q, double scale) {
  check_latent(qa, cache, bt);
  check_lens(seq_lens, bt);
  TORCH_CHECK(qa.scalar_type() == torch::kBFloat16);
  const long T = qa.size(0), H = qa.size(1), RP = qa.size(2), B = seq_lens.numel();
  on_gpu({cu});
  if (cu.has_value()) {
    TORCH_CHECK(cu->scalar_type() == torch::kInt && cu->is_contiguous() && cu->numel() == B + 1);
  } else {
    TORCH_CHECK(B == T && max_q == 1);
  }
  auto out = torch::empty_like(qa);
  if (T == 0) return out;
  const long units_x = (max_q * H + 15) / 16, units = units_x * B;
  LatentArgs a{};
  a.qa = (const short*)qa.data_ptr();
  a.cache = (const short*)cache.data_ptr();
  a.cu = cu.has_value() ? cu->data_ptr<int>() : nullptr;
  a.seq_lens = seq_lens.data_ptr<int>();
  a.bt = bt.data_ptr<int>();
  a.out = (short*)out.data_ptr();
  a.H = H;
  a.maxP = bt.size(1);
  a.scale = scale;
  // One workgroup per CU, none with less than two pages for every wave, all sequences with as
  // many parts.  Single tokens of long and uneven contexts divide all pages instead, which leaves
  // no CU idle and no context's parts longer than others.  How long they are is not known here, but
  // how many pages the table holds.  us, as many parts / all pages, of rows x mean of 512, lengths a
  // third to five thirds of it: 32 x 8000 64.6 / 55.4, 64 x 4000 64.0 / 58.5, 100 x 2600 74.2 / 56.8;
  // 100 of 60 and two of 16000 203 / 26, 48 of which 8 have 5000 41.1 / 40.9.  To find out takes a
  // workgroup 2 us and the merge 1, which short contexts in a wide table do not get back (2048
  // pages a row: 64 x 1000 23.9 / 24.4, 64 x 500 17.8 / 19.2, 32 x 500 12.4 / 15.5, 16 x 500 11.5 /
  // 14.7): up to 16 rows, which have 16 parts each anyway, only with 65536 pages.
  const long most = std::max<long>(1, bt.size(1) / 8), budget = 256 / units_x;
  a.splits = (int)std::min<long>(std::min<long>(most, 64), std::max<long>(1, 256 / units));
  a.B = B;
  a.budget = !cu.has_value() && B > 1 && 5 * B <= 2 * budget &&
                     B * units_x * bt.size(1) >= (B <= 16 ? 65536 : 16384) ? (int)budget : 0;
  torch::Tensor work;      // one allocation: the calls of small batches wait for the host
  if (a.splits > 1 || a.budget) {
    const long n = a.budget ? budget * units_x : units * a.splits;
    work = torch::empty({n * 16 * (RP + 2) + 2 * B}, qa.options().dtype(torch::kFloat32));
    a.part = work.data_ptr<float>();
    a.ms = a.part + n * 16 * RP;
    a.plan = (int2*)(a.ms + n * 32);
  }
  auto stream = at::hip::getCurrentHIPStream();
  TORCH_CHECK(B <= 65535, "too many sequences in a batch");
  const dim3 grid = a.budget ? dim3(units_x, budget) : dim3(units_x, B, a.splits);
#define LAUNCH(RR)                                                                            \
  do {                                                                                        \
    if (a.budget)                                                                             \
      hipLaunchKernelGGL((latent_attn_kernel<RR, true>), grid, dim3(256), 0, stream, a);      \
    else                                                                                      \
      hipLaunchKernelGGL((latent_attn_kernel<RR, false>), grid, dim3(256), 0, stream, a);     \
  } while (0)
  if (RP == 64) LAUNCH(64);
  else if (RP == 128) LAUNCH(128);
  else if (RP == 256) LAUNCH(256);
  else if (RP == 512) LAUNCH(512);
  else TORCH_CHECK(false, "unsupported latent width ", RP);
#undef LAUNCH
#define MERGE(MOST, ALL)                                                                      \
  hipLaunchKernelGGL((latent_merge_kernel<MOST, ALL>), dim3(units, 16), dim3(128), 0, stream, a,     \
                     (int)RP, (int)units_x)
  if (a.budget) MERGE(0, true);
  else if (a.splits > 4) MERGE(0, false);
  else if (a.splits > 1) MERGE(4, false);
#undef MERGE
  HIP_CHECK_LAST();
  return out;
}
