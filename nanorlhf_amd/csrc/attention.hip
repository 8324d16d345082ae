// Varlen causal flash attention, forward + backward, MFMA bf16 for gfx950.
//
// Sequences are packed ([T, H, D] with cu_seqlens); a workgroup of four waves
// owns 128 rows of one sequence and head, 32 per wave, and walks the other side
// in tiles of 64 rows, which two LDS buffers receive by direct loads
// (global_load_lds) while the tile before is computed on.
//
//   fa_fwd_kernel   rows of q; S^T = K Q^T, so a lane holds scores of ONE q
//                   row and the online softmax is lane-local; O^T += V^T P^T
//   fa_bwd_dq       rows of q; S^T and dP^T = V dO^T the same way, then
//                   dQ^T += K^T dS^T
//   fa_bwd_dkv      rows of k and v; S = Q K^T and dP = dO V^T, then
//                   dV += P^T dO and dK += dS^T Q over all q heads of the group
//
// The backward runs S and dP twice (7 products instead of 5) and in return
// has no atomics: dq, dk and dv are summed in registers in a fixed order and
// written once.
//
// What bounds them: the matrix products (0.47 of the forward's cycles, 0.58 of dq's, 0.51 of
// dk's and dv's, at 1.9 of 2.4 GHz), the VALU
// work between them (0.46, 0.37 and 0.28: an exponential, a fused multiply-add, an addition and
// half a conversion per score, and the fragments' addresses) and LDS reads (16 KB of
// fragments per 32 x 32 scores and two products).  Two waves per SIMD overlap the reads, but
// hardly the first two, whose shares add up to one in the forward of 64-wide heads.  5 causal sequences of about 6500 tokens, 12 heads over 2, width 128:
// forward 0.90 to 1.02 ms (830 to 940 TFLOP/s), backward 2.83; before, with V
// transposed by scalar LDS writes, 2.9 ms, and with dq added up by float atomics over
// 32-row kv tiles, 21.5 ms for the backward.  Twice the rows per wave (half the LDS
// reads, one wave per SIMD) and eight waves to a workgroup (half the loads) were slower
// everywhere; the next tile's scores under this one's exponentials, a part of two products at
// a time, took the same time.
//
// Products contract over the MFMA's k index in any order as long as both
// operands agree.  The C layout gives a lane the rows {0-3, 8-11} + 4 * half of
// each 16, so a P or dS fragment is those registers converted in place, and the
// other operand, a transposed LDS read of a row-major tile (ds_read_tr16_b64:
// 16 lanes, 4 rows x 16 columns), simply starts at the same rows.
//
// Replaces the reference's flash_attention_2 dependency
// (GRPO/grpo.py:219,223); packed varlen replaces its pad-mask forward
// (grpo_trainer.py:90-120).
#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>

#include <algorithm>

#include "common.h"
#include "lds_tiles.h"

constexpr float LOG2E = 1.4426950408889634f;
constexpr int ROWS = 128;    // rows that a workgroup owns, 32 per wave

// registers 8 * ks .. 8 * ks + 7 of a 32x32 result as a fragment of 16 rows
DEVINL bf16x8 pack_frag(const float* p) {
  union { unsigned u[4]; bf16x8 f; } fr;
#pragma unroll
  for (int j = 0; j < 4; j++) fr.u[j] = pack2bf(p[2 * j], p[2 * j + 1]);
  return fr.f;
}

// fragments of a row that stays in registers, along D
template <int D>
DEVINL void load_row(const short* __restrict__ p, int hi, bf16x8* f) {
#pragma unroll
  for (int ds = 0; ds < D / 16; ds++)
    f[ds] = *reinterpret_cast<const bf16x8*>(p + 16 * ds + 8 * hi);
}

DEVINL float other_half(float x, int hi) {
  auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(hi ? r[0] : r[1]);
}

// a lane's column of a transposed [D, 32] result as a bf16 row
template <int D>
DEVINL void store_row(short* __restrict__ dst, const f32x16_t* acc, float mul, int hi) {
#pragma unroll
  for (int c = 0; c < D / 32; c++)
#pragma unroll
    for (int g = 0; g < 4; g++) {
      union { unsigned u[2]; unsigned long long w; } o;
      o.u[0] = pack2bf(acc[c][4 * g] * mul, acc[c][4 * g + 1] * mul);
      o.u[1] = pack2bf(acc[c][4 * g + 2] * mul, acc[c][4 * g + 3] * mul);
      *reinterpret_cast<unsigned long long*>(dst + 32 * c + 8 * g + 4 * hi) = o.w;
    }
}

// Which sequence, head and tile a workgroup has.  `window` heads (of whichever sequences)
// are taken at a time, and of these tile first, the longest walks first: a causal row
// tile's work grows with its index, a kv tile's shrinks.  Workgroups go round the chiplets,
// of which each has its own L2, so a head stays with one if the window is a multiple of 8.
struct Place { int seq, head, s0, len, tile; };
template <bool LAST_FIRST>
DEVINL Place place(const int* __restrict__ cu, int heads, unsigned window) {
  const unsigned n = gridDim.x, tiles = gridDim.y;
  unsigned x = blockIdx.x, y = blockIdx.y;
  if (window < n) {
    const unsigned at = y * n + x, begin = at / (window * tiles) * window;
    const unsigned wide = min(window, n - begin), in = at - begin * tiles;
    x = begin + in % wide;
    y = in / wide;
  }
  Place p;
  p.seq = x / heads;
  p.head = x % heads;
  p.s0 = cu[p.seq];
  p.len = cu[p.seq + 1] - p.s0;
  p.tile = LAST_FIRST ? tiles - 1 - y : y;
  return p;
}

// ================================================================ FORWARD ==
template <int D, bool CAUSAL>
__global__ __launch_bounds__(256, 2)
void fa_fwd_kernel(const short* __restrict__ q, const short* __restrict__ k,
                   const short* __restrict__ v, const int* __restrict__ cu,
                   short* __restrict__ o, float* __restrict__ lse, int Hq, int Hkv, float scale,
                   unsigned window) {
  constexpr int NDS = D / 16, NDT = D / 32;
  constexpr float THR = 11.54f;       // rescale when a row grows past 8 nats (log2 units)
  const Place pl = place<CAUSAL>(cu, Hq, window);
  const int len = pl.len, h = pl.head, kvh = h / (Hq / Hkv);
  const int q0 = pl.tile * ROWS;
  if (q0 >= len) return;
  const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int hi = lane >> 5;
  const int qw0 = q0 + wid * 32, qi = qw0 + (lane & 31);

  __shared__ short lds[2][2][TILE * D];   // [buffer][K, V]

  bf16x8 qf[NDS];
  load_row<D>(q + ((long)(pl.s0 + min(qi, len - 1)) * Hq + h) * D, hi, qf);
  float m = -INFINITY, sum = 0.f;
  f32x16_t acc[NDT];
#pragma unroll
  for (int c = 0; c < NDT; c++) acc[c] = f32x16_t{};
  const int ld = Hkv * D;
  const short* kb = k + (long)pl.s0 * ld + kvh * D;
  const short* vb = v + (long)pl.s0 * ld + kvh * D;
  const int kv_end = CAUSAL ? min(len, q0 + ROWS) : len;
  const int kv_end_w = qw0 >= len ? 0 : CAUSAL ? min(len, qw0 + 32) : len;
  const float sl2 = scale * LOG2E;

  stage_tile<D>(kb, ld, len, lds[0][0]);
  stage_tile<D>(vb, ld, len, lds[0][1]);
  int buf = 0;
  for (int kv0 = 0; kv0 < kv_end; kv0 += TILE, buf ^= 1) {
    tiles_ready();
    if (kv0 + TILE < kv_end) {
      stage_tile<D>(kb + (long)(kv0 + TILE) * ld, ld, len - kv0 - TILE, lds[buf ^ 1][0]);
      stage_tile<D>(vb + (long)(kv0 + TILE) * ld, ld, len - kv0 - TILE, lds[buf ^ 1][1]);
    }
    if (kv0 >= kv_end_w) continue;
    const short* Kt = lds[buf][0];
    const short* Vt = lds[buf][1];

    f32x16_t st[2];
#pragma unroll
    for (int sub = 0; sub < 2; sub++) {
      st[sub] = f32x16_t{};
#pragma unroll
      for (int ds = 0; ds < NDS; ds++)
        st[sub] = mfma32x32x16(row_frag<D>(Kt, 32 * sub, ds, lane), qf[ds], st[sub]);
    }
    // Scores stay as they are and meet scale * log2(e) in the exponent's fma
    // (the softmax runs in base 2), which needs a positive scale.
    float mul = sl2;
    if (!(sl2 > 0.f)) {
#pragma unroll
      for (int r = 0; r < 32; r++) st[r >> 4][r & 15] *= sl2;
      mul = 1.f;
    }
    if (!(kv0 + TILE <= len && (!CAUSAL || kv0 + TILE - 1 <= qw0))) {
#pragma unroll
      for (int r = 0; r < 32; r++) {
        const int ki = kv0 + 32 * (r >> 4) + crow(r & 15, hi);
        if (!(ki < len && (!CAUSAL || ki <= qi))) st[r >> 4][r & 15] = -INFINITY;
      }
    }
    float top = st[0][0];
#pragma unroll
    for (int r = 1; r < 32; r++) top = fmaxf(top, st[r >> 4][r & 15]);
    top = fmaxf(top, other_half(top, hi)) * mul;
    // rescale only when some row grew past THR (or has no maximum yet)
    float alpha = 1.f;
    if (__any(!(top - m <= THR))) {
      const float mn = fmaxf(m, top);
      alpha = (m == -INFINITY) ? 0.f : exp2f(m - mn);
      m = mn;
#pragma unroll
      for (int c = 0; c < NDT; c++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[c][r] *= alpha;
    }
    const float mm = m == -INFINITY ? 0.f : m;   // a row that sees nothing so far
    float p[32], rs = 0.f;
#pragma unroll
    for (int r = 0; r < 32; r++) {
      p[r] = __builtin_amdgcn_exp2f(fmaf(st[r >> 4][r & 15], mul, -mm));
      rs += p[r];
    }
    sum = sum * alpha + rs + other_half(rs, hi);
#pragma unroll
    for (int ks = 0; ks < 4; ks++) {
      const bf16x8 pf = pack_frag(p + 8 * ks);
#pragma unroll
      for (int c = 0; c < NDT; c++)
        acc[c] = mfma32x32x16(col_frag<D>(Vt, 16 * ks, 32 * c, lane), pf, acc[c]);
    }
  }
  if (qi >= len) return;
  store_row<D>(o + ((long)(pl.s0 + qi) * Hq + h) * D, acc, sum > 0.f ? 1.f / sum : 0.f, hi);
  if (hi == 0)   // m is in log2 units: lse = ln2 * (m + log2 s)
    lse[(long)(pl.s0 + qi) * Hq + h] = 0.6931471805599453f * (m + log2f(fmaxf(sum, 1e-30f)));
}

// =============================================================== BACKWARD ==
// rows [Hq, T]: -sum(dO * O), which dP starts from in the matrix product's
// accumulator, and lse in log2 units.  16 lanes per row.  Tokens ahead of the first
// sequence and behind the last (padding) have no gradient: nobody else writes theirs.
DEVINL bool outside(long t, const int* __restrict__ cu, int B) { return t < cu[0] || t >= cu[B]; }
template <int D>
__global__ __launch_bounds__(256)
void fa_bwd_rows_kernel(const short* __restrict__ dout, const short* __restrict__ o,
                        const float* __restrict__ lse, float* __restrict__ drow,
                        float* __restrict__ lse2, const int* __restrict__ cu, int B,
                        short* __restrict__ dq, short* __restrict__ dk, short* __restrict__ dv,
                        long T, int Hq, int Hkv) {
  const long row = (long)blockIdx.x * 16 + (threadIdx.x >> 4);   // t * Hq + h
  const int i = threadIdx.x & 15;
  float acc = 0.f;
  if (row < T * Hq) {
    float a[D / 16], b[D / 16];
    ldv<D / 16>(dout + row * D + i * (D / 16), a);
    ldv<D / 16>(o + row * D + i * (D / 16), b);
#pragma unroll
    for (int j = 0; j < D / 16; j++) acc += a[j] * b[j];
    const long t = row / Hq, h = row % Hq;
    if (outside(t, cu, B)) {
      const float zero[D / 16] = {};
      stv<D / 16>(dq + row * D + i * (D / 16), zero);
      if (h < Hkv) {
        const long at = (t * Hkv + h) * D + i * (D / 16);
        stv<D / 16>(dk + at, zero);
        stv<D / 16>(dv + at, zero);
      }
    }
  }
#pragma unroll
  for (int off = 8; off > 0; off >>= 1) acc += __shfl_xor(acc, off);
  if (i == 0 && row < T * Hq) {
    const long at = (row % Hq) * T + row / Hq;
    drow[at] = -acc;
    lse2[at] = lse[row] * LOG2E;
  }
}

template <int D, bool CAUSAL>
__global__ __launch_bounds__(256, 2)
void fa_bwd_dq_kernel(const short* __restrict__ dout, const short* __restrict__ q,
                      const short* __restrict__ k, const short* __restrict__ v,
                      const float* __restrict__ lse2, const float* __restrict__ drow,
                      const int* __restrict__ cu, short* __restrict__ dq, long T, int Hq,
                      int Hkv, float scale, unsigned window) {
  constexpr int NDS = D / 16, NDT = D / 32;
  const Place pl = place<CAUSAL>(cu, Hq, window);
  const int len = pl.len, h = pl.head, kvh = h / (Hq / Hkv);
  const int q0 = pl.tile * ROWS;
  if (q0 >= len) return;
  const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int hi = lane >> 5;
  const int qw0 = q0 + wid * 32, qi = qw0 + (lane & 31), qc = min(qi, len - 1);

  __shared__ short lds[2][2][TILE * D];   // [buffer][K, V]

  bf16x8 qf[NDS], dof[NDS];
  const long base = ((long)(pl.s0 + qc) * Hq + h) * D;
  load_row<D>(q + base, hi, qf);
  load_row<D>(dout + base, hi, dof);
  const float l2 = lse2[(long)h * T + pl.s0 + qc], dr = drow[(long)h * T + pl.s0 + qc];
  f32x16_t acc[NDT];
#pragma unroll
  for (int c = 0; c < NDT; c++) acc[c] = f32x16_t{};
  const int ld = Hkv * D;
  const short* kb = k + (long)pl.s0 * ld + kvh * D;
  const short* vb = v + (long)pl.s0 * ld + kvh * D;
  const int kv_end = CAUSAL ? min(len, q0 + ROWS) : len;
  const int kv_end_w = qw0 >= len ? 0 : CAUSAL ? min(len, qw0 + 32) : len;
  const float sl2 = scale * LOG2E;

  stage_tile<D>(kb, ld, len, lds[0][0]);
  stage_tile<D>(vb, ld, len, lds[0][1]);
  int buf = 0;
  for (int kv0 = 0; kv0 < kv_end; kv0 += TILE, buf ^= 1) {
    tiles_ready();
    if (kv0 + TILE < kv_end) {
      stage_tile<D>(kb + (long)(kv0 + TILE) * ld, ld, len - kv0 - TILE, lds[buf ^ 1][0]);
      stage_tile<D>(vb + (long)(kv0 + TILE) * ld, ld, len - kv0 - TILE, lds[buf ^ 1][1]);
    }
    const short* Kt = lds[buf][0];
    const short* Vt = lds[buf][1];
#pragma unroll
    for (int sub = 0; sub < 2; sub++) {
      const int kv1 = kv0 + 32 * sub;
      if (kv1 >= kv_end_w) continue;
      f32x16_t st{}, dp;
#pragma unroll
      for (int r = 0; r < 16; r++) dp[r] = dr;
#pragma unroll
      for (int ds = 0; ds < NDS; ds++) {
        st = mfma32x32x16(row_frag<D>(Kt, 32 * sub, ds, lane), qf[ds], st);
        dp = mfma32x32x16(row_frag<D>(Vt, 32 * sub, ds, lane), dof[ds], dp);
      }
      float s[16];
#pragma unroll
      for (int r = 0; r < 16; r++)
        s[r] = __builtin_amdgcn_exp2f(fmaf(st[r], sl2, -l2)) * dp[r];
      if (!(kv1 + 32 <= len && (!CAUSAL || kv1 + 31 <= qw0))) {
#pragma unroll
        for (int r = 0; r < 16; r++) {
          const int ki = kv1 + crow(r, hi);
          if (!(ki < len && (!CAUSAL || ki <= qi))) s[r] = 0.f;
        }
      }
#pragma unroll
      for (int ks = 0; ks < 2; ks++) {
        const bf16x8 sf = pack_frag(s + 8 * ks);
#pragma unroll
        for (int c = 0; c < NDT; c++)
          acc[c] = mfma32x32x16(col_frag<D>(Kt, 32 * sub + 16 * ks, 32 * c, lane), sf, acc[c]);
      }
    }
  }
  if (qi < len) store_row<D>(dq + ((long)(pl.s0 + qi) * Hq + h) * D, acc, scale, hi);
}

// blockIdx.x = (sequence, kv head, part); part p of `parts` sums over its share
// of the group's q heads.  One part writes bf16 (dk, dv); several write float
// partial sums [parts, T, Hkv, D] into dk, dv.
template <int D, bool CAUSAL>
__global__ __launch_bounds__(256, 2)
void fa_bwd_dkv_kernel(const short* __restrict__ dout, const short* __restrict__ q,
                       const short* __restrict__ k, const short* __restrict__ v,
                       const float* __restrict__ lse2, const float* __restrict__ drow,
                       const int* __restrict__ cu, void* __restrict__ dk,
                       void* __restrict__ dv, long T, int Hq, int Hkv, int parts, float scale,
                       unsigned window) {
  constexpr int NDS = D / 16, NDT = D / 32;
  const Place pl = place<false>(cu, Hkv * parts, window);
  const int len = pl.len, kvh = pl.head / parts, part = pl.head % parts;
  const int heads = Hq / Hkv / parts, h0 = kvh * (Hq / Hkv) + part * heads;
  const int kv0 = pl.tile * ROWS;
  if (kv0 >= len) return;
  const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int hi = lane >> 5;
  const int kw0 = kv0 + wid * 32, ki = kw0 + (lane & 31);

  __shared__ __attribute__((aligned(256))) short lds[2][2][TILE * D];   // [buffer][Q, dO]
  __shared__ float rows[2][2][TILE];      // [buffer][lse2, -sum(dO * O)]

  bf16x8 kf[NDS], vf[NDS];
  const long base = ((long)(pl.s0 + min(ki, len - 1)) * Hkv + kvh) * D;
  load_row<D>(k + base, hi, kf);
  load_row<D>(v + base, hi, vf);
  f32x16_t adk[NDT], adv[NDT];
#pragma unroll
  for (int c = 0; c < NDT; c++) adk[c] = adv[c] = f32x16_t{};
  const int ld = Hq * D;
  const int qstart = CAUSAL ? kv0 / TILE * TILE : 0;
  const float sl2 = scale * LOG2E;
  const bool wave_active = kw0 < len;

  // (lse2 and drow too: through a register they would be waited for behind the tiles)
  auto stage = [&](int h, int r0, int buf) {
    const long at = (long)(pl.s0 + r0) * ld + h * D;
    stage_tile<D>(q + at, ld, len - r0, lds[buf][0]);
    stage_tile<D>(dout + at, ld, len - r0, lds[buf][1]);
    if (wid < 2)
      load_to_lds4((wid ? drow : lse2) + (long)h * T + pl.s0 + r0, 4 * min(lane, len - r0 - 1),
                   rows[buf][wid]);
  };
  constexpr unsigned BUFFER = sizeof(lds[0]);     // dO's tile lies TILE rows behind Q's
  const unsigned base0 = lds_address(&lds[0][0][0]);
  const unsigned row0 = base0 + row_at<D>(lane), col0 = base0 + col_at<D>(lane);
  stage(h0, qstart, 0);
  int h = h0, r0 = qstart, buf = 0;
  for (; h < h0 + heads; buf ^= 1) {
    tiles_ready();
    int hn = h, rn = r0 + TILE;
    if (rn >= len) { hn++; rn = qstart; }
    if (hn < h0 + heads) stage(hn, rn, buf ^ 1);
#pragma unroll
    for (int sub = 0; sub < 2; sub++) {
      const int q1 = r0 + 32 * sub;
      if (!wave_active || q1 >= len || (CAUSAL && q1 + 31 < kw0)) continue;
      const bool whole = q1 + 32 <= len && (!CAUSAL || kw0 + 31 <= q1);
      // K, V and the sums fill the registers: two addresses are kept, the others made
      // from them each time and phases kept apart, or fragments go to scratch memory
      unsigned ra = row0 + buf * BUFFER, ca = col0 + buf * BUFFER;
      asm volatile("" : "+v"(ra), "+v"(ca));
      f32x16_t st{}, dp;
#pragma unroll
      for (int g = 0; g < 4; g++)
#pragma unroll
        for (int j = 0; j < 4; j++) dp[4 * g + j] = rows[buf][1][32 * sub + 8 * g + 4 * hi + j];
#pragma unroll
      for (int ds = 0; ds < NDS; ds++)
        st = mfma32x32x16(row_frag_at<D>(ra, 32 * sub, ds), kf[ds], st);
#pragma unroll
      for (int ds = 0; ds < NDS; ds++)
        dp = mfma32x32x16(row_frag_at<D>(ra, TILE + 32 * sub, ds), vf[ds], dp);
      __builtin_amdgcn_sched_barrier(0);
      float p[16], s[16];
#pragma unroll
      for (int g = 0; g < 4; g++) {
        const int at = 32 * sub + 8 * g + 4 * hi;
        const f32x4 l4 = *reinterpret_cast<const f32x4*>(&rows[buf][0][at]);
#pragma unroll
        for (int j = 0; j < 4; j++) {
          const int r = 4 * g + j;
          p[r] = __builtin_amdgcn_exp2f(fmaf(st[r], sl2, -l4[j]));
          s[r] = p[r] * dp[r];
        }
      }
      if (!whole) {
#pragma unroll
        for (int r = 0; r < 16; r++) {
          const int qi = q1 + crow(r, hi);
          if (!(qi < len && (!CAUSAL || ki <= qi))) p[r] = s[r] = 0.f;
        }
      }
#pragma unroll
      for (int ks = 0; ks < 2; ks++) {
        __builtin_amdgcn_sched_barrier(0);
        const bf16x8 pf = pack_frag(p + 8 * ks), sf = pack_frag(s + 8 * ks);
#pragma unroll
        for (int c = 0; c < NDT; c++) {
          const int r = 32 * sub + 16 * ks;
          adv[c] = mfma32x32x16(pf, col_frag_at<D>(ca, TILE + r, 32 * c), adv[c]);
          adk[c] = mfma32x32x16(sf, col_frag_at<D>(ca, r, 32 * c), adk[c]);
        }
      }
    }
    h = hn;
    r0 = rn;
  }
#pragma unroll
  for (int r = 0; r < 16; r++) {
    const int kr = kw0 + crow(r, hi);
    if (kr >= len) continue;
    const long at = (((long)part * T + pl.s0 + kr) * Hkv + kvh) * D + (lane & 31);
#pragma unroll
    for (int c = 0; c < NDT; c++) {
      if (parts == 1) {
        ((short*)dk)[at + 32 * c] = f2bf(adk[c][r] * scale);
        ((short*)dv)[at + 32 * c] = f2bf(adv[c][r]);
      } else {
        ((float*)dk)[at + 32 * c] = adk[c][r] * scale;
        ((float*)dv)[at + 32 * c] = adv[c][r];
      }
    }
  }
}

// sums of the parts, in order; n elements each, 4 per thread, `width` per token; y = 0:
// dk, 1: dv
__global__ void fa_bwd_sum_kernel(const float* __restrict__ part, short* __restrict__ dk,
                                  short* __restrict__ dv, const int* __restrict__ cu, int B,
                                  long n, int width, int parts) {
  const long i = ((long)blockIdx.x * blockDim.x + threadIdx.x) * 4;
  if (i >= n || outside(i / width, cu, B)) return;
  const float* p = part + (blockIdx.y ? (long)parts * n : 0) + i;
  f32x4 s = *reinterpret_cast<const f32x4*>(p);
  for (int k = 1; k < parts; k++) s += *reinterpret_cast<const f32x4*>(p + k * n);
  s16x4 o;
#pragma unroll
  for (int j = 0; j < 4; j++) o[j] = f2bf(s[j]);
  *reinterpret_cast<s16x4*>((blockIdx.y ? dv : dk) + i) = o;
}

// ======================================================== host wrappers ==
// Heads that workgroups are taken from at a time.  As many as fill every chiplet's 32 CUs
// twice: what runs there together then shares the tiles that its L2 holds.  Or all, so that
// the longest walks of all come first, which a causal grid needs to end evenly unless it is
// several rounds of the workgroups that run at a time and the last window, which may hold the
// longest sequence, is a small part of it.  Forward, all heads / a window, us:
// 80 x 800 not causal, 16 heads of 64 456 / 371 (70% of the tiles' requests missed the L2);
// causal, 12 heads over 2 of 128: 56 x 870 256 / 221, 16 x 1500 194 / 167, 16 x 6000 2550 /
// 2050; 3.5 rounds, 28 heads over 4, 4 x 2000 139 / 146; 2.8 rounds, 14 heads of 64, 20 x
// 1200 102 / 121; 7.5 windows, 5 x 6500 896 / 880 with the longest sequence ahead, but forward
// and backward 3811 / 3997 with it behind.  Backward of the first 1354 / 1118.  The walks of
// dk and dv are few and long: causal, 40 x 1200 1041 / 1291.  The forward of up to two tiles
// has little to share before it ends: not causal, 16 heads of 64, 64 x 100 18.7 / 20.5, 12 of
// 128 27.8 / 28.8; with 3.9 rounds, 128 x 120, 40.0 / 37.5.  A window's place is found from
// the workgroup's number, which has to fit 32 bits.
long fa_head_window(long heads, long tiles, long rounds, bool causal) {
  const long window = 8 * std::max(64 / std::max(tiles, 1L), 1L);
  return causal && (rounds < 4 || heads < 8 * window) || heads * tiles >= 1L << 32 ? heads : window;
}

#define FA_BY_WIDTH(CALL)                                                  \
  do {                                                                     \
    if (D == 128) { if (causal) CALL(128, true); else CALL(128, false); }  \
    else if (D == 64) { if (causal) CALL(64, true); else CALL(64, false); } \
    else if (D == 32) { if (causal) CALL(32, true); else CALL(32, false); } \
    else TORCH_CHECK(false, "unsupported head_dim ", D);                   \
  } while (0)

std::vector<torch::Tensor> fa_fwd_varlen(torch::Tensor q, torch::Tensor k,
                                         torch::Tensor v, torch::Tensor cu_seqlens,
                                         long max_seqlen, double scale, bool causal) {
  TORCH_CHECK(q.scalar_type() == torch::kBFloat16 && q.is_contiguous());
  TORCH_CHECK(cu_seqlens.scalar_type() == torch::kInt);
  const long T = q.size(0);
  const int Hq = q.size(1), D = q.size(2), Hkv = k.size(1);
  const int B = cu_seqlens.size(0) - 1;
  auto o = torch::empty_like(q);
  auto lse = torch::empty({T, Hq}, q.options().dtype(torch::kFloat32));
  if (T == 0) return {o, lse};
  auto stream = at::hip::getCurrentHIPStream();
  const dim3 grid(B * Hq, (max_seqlen + ROWS - 1) / ROWS);
  const long rounds = (T / ROWS + B) * Hq / (D > 64 ? 512 : 1024);
  const bool short_walks = grid.y <= 2 && rounds < 3;
#define CALL(DD, CC)                                                           \
  hipLaunchKernelGGL((fa_fwd_kernel<DD, CC>), grid, dim3(256), 0, stream,      \
                     (const short*)q.data_ptr(), (const short*)k.data_ptr(),   \
                     (const short*)v.data_ptr(), cu_seqlens.data_ptr<int>(),   \
                     (short*)o.data_ptr(), lse.data_ptr<float>(), Hq, Hkv, (float)scale,     \
                     fa_head_window(grid.x, grid.y, rounds, causal || short_walks))
  FA_BY_WIDTH(CALL);
#undef CALL
  HIP_CHECK_LAST();
  return {o, lse};
}

// A workgroup of dk and dv walks the group's q heads one after the other.  Where that leaves
// too few to fill 256 CUs twice, with spare to even out causal tiles, they are divided among
// `parts`.  Long sequences want more of them the shorter the others are, for a walk of the
// longest then is more of the whole, and with heads of 64, of which a CU runs more
// at a time.  From 1100 undivided ones on there is one part, which bounds the parts'
// memory.  Whole backward, us by parts, undivided workgroups in brackets:
//   12 heads over 2   56 x 870 (872) 1: 720, 2: 770, 6: 890   8 x 3000 (390) 2: 1130, 3: 1160
//     equal lengths   2 x 6000 (190) 3: 854, 6: 762   3 x 6000 (286) 2: 1260, 3: 1114, 6: 1131
//                     4 x 6000 (382) 2: 1485, 3: 1450   5 x 6000 (478) 2: 1845, 3: 1848
//     mixed           8000 2 x, 3000 6 x (546) 2: 3021, 3: 2071   7900, 600 30 x (466) 2: 1441, 3: 1238
//     up to 10000     5 of 6900 (546) 1: 3971, 2: 2888, 3: 2887
//   28 heads over 4   5 x 6000 (956) 1: 4319, 7: 4555   4 x 8000 (1016) 1: 6019, 7: 6146
//     mixed           4 of 6200 (796) 1: 5743, 7: 4601   7900, 600 30 x (932) 1: 3179, 7: 2239
//     up to 10000     5 of 6900 (1092) 1: 6782, 7: 7134
//   14 over 2 of 64   9 x 6000 (860) 1: 2265, 7: 2092   8 x 8000 (1016) 1: 3241, 7: 3153
//                     12 x 6000 (1148) 1: 2652, 7: 2758
long fa_bwd_parts(long T, long B, long Hq, long Hkv, long D, long max_seqlen) {
  const long G = Hq / Hkv, tiles = (T / ROWS + B) * Hkv;
  const long wanted = max_seqlen < 6000 ? 768
                      : D <= 64         ? 1100
                                        : std::clamp(720 * max_seqlen * B / T, 768L, 1100L);
  long parts = 1;
  while (parts < G && (G % parts || tiles * parts < wanted)) parts++;
  return parts;
}

std::vector<torch::Tensor> fa_bwd_varlen(torch::Tensor dout, torch::Tensor q,
                                         torch::Tensor k, torch::Tensor v,
                                         torch::Tensor o, torch::Tensor lse,
                                         torch::Tensor cu_seqlens, long max_seqlen,
                                         double scale, bool causal) {
  TORCH_CHECK(dout.scalar_type() == torch::kBFloat16 && dout.is_contiguous());
  const long T = q.size(0);
  const int Hq = q.size(1), D = q.size(2), Hkv = k.size(1), G = Hq / Hkv;
  const int B = cu_seqlens.size(0) - 1;
  auto dq = torch::empty_like(q), dk = torch::empty_like(k), dv = torch::empty_like(v);
  if (T == 0) return {dq, dk, dv};
  auto f32 = q.options().dtype(torch::kFloat32);
  auto rows = torch::empty({2, (long)Hq, T}, f32);    // -sum(dO * O), lse in log2 units
  float* drow = rows.data_ptr<float>();
  float* lse2 = drow + (long)Hq * T;
  const int parts = fa_bwd_parts(T, B, Hq, Hkv, D, max_seqlen);
  const long n = T * Hkv * D;
  torch::Tensor sums;
  if (parts > 1) sums = torch::empty({2, (long)parts, n}, f32);
  void* dkp = parts > 1 ? (void*)sums.data_ptr<float>() : dk.data_ptr();
  void* dvp = parts > 1 ? (void*)(sums.data_ptr<float>() + parts * n) : dv.data_ptr();
  auto stream = at::hip::getCurrentHIPStream();
  const int row_tiles = (max_seqlen + ROWS - 1) / ROWS;
  const long rounds = (T / ROWS + B) * Hq / (D > 64 ? 512 : 1024);
#define CALL(DD, CC)                                                           \
  do {                                                                         \
    hipLaunchKernelGGL(fa_bwd_rows_kernel<DD>, dim3((T * Hq + 15) / 16), dim3(256), 0, stream, \
                       (const short*)dout.data_ptr(), (const short*)o.data_ptr(), \
                       lse.data_ptr<float>(), drow, lse2, cu_seqlens.data_ptr<int>(), B, \
                       (short*)dq.data_ptr(), (short*)dk.data_ptr(), (short*)dv.data_ptr(), T, \
                       Hq, Hkv);                                               \
    hipLaunchKernelGGL((fa_bwd_dq_kernel<DD, CC>), dim3(B * Hq, row_tiles), dim3(256), 0, stream, \
                       (const short*)dout.data_ptr(), (const short*)q.data_ptr(), \
                       (const short*)k.data_ptr(), (const short*)v.data_ptr(), \
                       lse2, drow, cu_seqlens.data_ptr<int>(), (short*)dq.data_ptr(), \
                       T, Hq, Hkv, (float)scale,                               \
                       fa_head_window(B * Hq, row_tiles, rounds, causal));     \
    hipLaunchKernelGGL((fa_bwd_dkv_kernel<DD, CC>), dim3(B * Hkv * parts, row_tiles), dim3(256), \
                       0, stream, (const short*)dout.data_ptr(),               \
                       (const short*)q.data_ptr(), (const short*)k.data_ptr(), \
                       (const short*)v.data_ptr(), lse2, drow,                 \
                       cu_seqlens.data_ptr<int>(), dkp, dvp, T, Hq, Hkv, parts, (float)scale, \
                       fa_head_window(B * Hkv * parts, row_tiles, 0, causal)); \
  } while (0)
  FA_BY_WIDTH(CALL);
#undef CALL
  if (parts > 1)
    hipLaunchKernelGGL(fa_bwd_sum_kernel, dim3((n / 4 + 255) / 256, 2), dim3(256), 0, stream,
                       sums.data_ptr<float>(), (short*)dk.data_ptr(), (short*)dv.data_ptr(),
                       cu_seqlens.data_ptr<int>(), B, n, (int)(Hkv * D), parts);
  HIP_CHECK_LAST();
  return {dq, dk, dv};
}
