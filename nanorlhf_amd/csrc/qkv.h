// A layer's q, k and v leave their projection: rows [Hq + 2 Hkv heads][D] are
// split, q and k rotated (rotate-half), k and v written to the paged cache if
// there is one.  One pass over the projection, where three copies, two rotations
// and an append each took a launch.
//
// One thread moves 16 bytes from either half of a head: 8 pairs of q or k, or 16
// elements of v.  Bound by memory, or by the launch when decoding: a rollout of 64
// rows and 96 tokens through 6 layers went from 95 to 86 ms.
#pragma once

#include <hip/hip_runtime.h>

#include "common.h"

struct QkvRope {
  const short* qkv;      // [T, Hq + 2 Hkv, D]
  short *q, *k, *v;      // [T, Hq, D], [T, Hkv, D]; k and v may be null
  const float* table;    // [maxpos, D] cos | sin halves
  const long* pos;       // [T]
  const long* slots;     // [T] flat cache slots, with a cache
  void *kc, *vc;         // [P, ps, Hkv, D], [P, Hkv, D, ps]
  int Hq, Hkv, D, ps;
  // instead of qkv: 32-bit sums of parts of the projection's depth [splits][T, ..] and bias
  const float* parts;
  const short* bias;     // may be null
  long part;             // elements of one
  int splits;
};

DEVINL void rotate8(const s16x8& x1, const s16x8& x2, const float* tb, int D, float sign, s16x8& o1,
                    s16x8& o2) {
  float c[8], s[8];
  ldv<8>(tb, c);
  ldv<8>(tb + D / 2, s);
#pragma unroll
  for (int j = 0; j < 8; j++) {
    const float a = bf2f(x1[j]), b = bf2f(x2[j]), sn = s[j] * sign;
    o1[j] = f2bf(a * c[j] - b * sn);
    o2[j] = f2bf(b * c[j] + a * sn);
  }
}

DEVINL unsigned fp8x4(const s16x8& x, int at) {
  unsigned w = __builtin_amdgcn_cvt_pk_fp8_f32(bf2f(x[at]), bf2f(x[at + 1]), 0, false);
  return __builtin_amdgcn_cvt_pk_fp8_f32(bf2f(x[at + 2]), bf2f(x[at + 3]), w, true);
}

// CT: element of the cache, or void
template <typename CT, bool PARTS = false>
__global__ __launch_bounds__(256) void qkv_rope_kernel(QkvRope a, unsigned units) {
  const unsigned idx = blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= units) return;
  const unsigned G = a.D / 16, H = a.Hq + 2 * a.Hkv;
  const unsigned g = idx % G, row = idx / G;       // row = t * H + h
  const unsigned h = row % H;
  const long t = row / H;
  // With a cache asked for first: few rows are a chain of loads (64 rows of 2048, cached, 2.98 us
  // and 3.17 asked for where they are needed).  Without one rows are many and the heads of v
  // need none: 5000 rows of 4608 16.7 us, 17.7 asked for first, 46673 of 2048 68.6 and 71.7.
  constexpr bool FIRST = !std::is_void_v<CT>;
  // The slot stays under a test that a cache always passes, for the order that the compiler then
  // gives the loads: 2000 rows of 4608 13.5 us, 14.9 without it.
  const long pos = FIRST ? a.pos[t] : 0, slot = a.slots ? a.slots[t] : 0;
  const int d1 = 8 * g, d2 = a.D / 2 + 8 * g;
  s16x8 x1, x2;
  if constexpr (PARTS) {
    const float* src = a.parts + (long)row * a.D;
    const short* bias = a.bias ? a.bias + h * a.D : nullptr;
    x1 = sum_parts8(src + d1, a.part, a.splits, bias ? bias + d1 : nullptr);
    x2 = sum_parts8(src + d2, a.part, a.splits, bias ? bias + d2 : nullptr);
  } else {
    const short* src = a.qkv + (long)row * a.D;
    x1 = *reinterpret_cast<const s16x8*>(src + d1);
    x2 = *reinterpret_cast<const s16x8*>(src + d2);
  }
  const bool is_v = h >= (unsigned)(a.Hq + a.Hkv), is_q = h < (unsigned)a.Hq;
  if (!is_v) rotate8(x1, x2, a.table + (FIRST ? pos : a.pos[t]) * a.D + d1, a.D, 1.f, x1, x2);
  const int kvh = is_v ? h - a.Hq - a.Hkv : (int)h - a.Hq;
  short* out = is_q ? a.q + (t * a.Hq + h) * a.D
                    : (is_v ? a.v : a.k) ? (is_v ? a.v : a.k) + (t * a.Hkv + kvh) * a.D : nullptr;
  if (out) {
    *reinterpret_cast<s16x8*>(out + d1) = x1;
    *reinterpret_cast<s16x8*>(out + d2) = x2;
  }
  if constexpr (!std::is_void_v<CT>) {
    if (is_q) return;
    if (!is_v) {
      CT* kc = (CT*)a.kc + (slot * a.Hkv + kvh) * a.D;
      if constexpr (sizeof(CT) == 2) {
        *reinterpret_cast<s16x8*>(kc + d1) = x1;
        *reinterpret_cast<s16x8*>(kc + d2) = x2;
      } else {
        // fragment-major: the 8 elements at d lie at (d % 32) / 8 * D / 4 + d / 32 * 8
        const int at1 = ((d1 >> 3) & 3) * (a.D >> 2) + (d1 >> 5) * 8;
        const int at2 = ((d2 >> 3) & 3) * (a.D >> 2) + (d2 >> 5) * 8;
        *reinterpret_cast<uint2*>(kc + at1) = make_uint2(fp8x4(x1, 0), fp8x4(x1, 4));
        *reinterpret_cast<uint2*>(kc + at2) = make_uint2(fp8x4(x2, 0), fp8x4(x2, 4));
      }
    } else {
      const long page = slot / a.ps;
      CT* vc = (CT*)a.vc + ((page * a.Hkv + kvh) * a.D) * a.ps + slot % a.ps;
#pragma unroll
      for (int j = 0; j < 8; j++) {
        if constexpr (sizeof(CT) == 2) {
          vc[(long)(d1 + j) * a.ps] = x1[j];
          vc[(long)(d2 + j) * a.ps] = x2[j];
        } else {
          vc[(long)(d1 + j) * a.ps] = (CT)(fp8x4(x1, j & 4) >> (8 * (j & 3)));
          vc[(long)(d2 + j) * a.ps] = (CT)(fp8x4(x2, j & 4) >> (8 * (j & 3)));
        }
      }
    }
  }
}

// gradients [T, Hq, D], [T, Hkv, D] x 2 (any may be null: zero) -> [T, Hq + 2 Hkv, D]
inline __global__ __launch_bounds__(256) void qkv_rope_bwd_kernel(
    const short* __restrict__ dq, const short* __restrict__ dk, const short* __restrict__ dv,
    const float* __restrict__ table, const long* __restrict__ pos, short* __restrict__ dqkv, int Hq,
    int Hkv, int D, unsigned units) {
  const unsigned idx = blockIdx.x * 256u + threadIdx.x;
  if (idx >= units) return;
  const unsigned G = D / 16, H = Hq + 2 * Hkv;
  const unsigned g = idx % G, row = idx / G;
  const unsigned h = row % H;
  const long t = row / H;
  const int d1 = 8 * g, d2 = D / 2 + 8 * g;
  const short* src = h < (unsigned)Hq ? dq : h < (unsigned)(Hq + Hkv) ? dk : dv;
  const long at = h < (unsigned)Hq ? t * Hq + h
                                   : t * Hkv + (h < (unsigned)(Hq + Hkv) ? h - Hq : h - Hq - Hkv);
  s16x8 x1{}, x2{};
  if (src) {
    x1 = *reinterpret_cast<const s16x8*>(src + at * D + d1);
    x2 = *reinterpret_cast<const s16x8*>(src + at * D + d2);
    if (h < (unsigned)(Hq + Hkv)) rotate8(x1, x2, table + pos[t] * D + d1, D, -1.f, x1, x2);
  }
  *reinterpret_cast<s16x8*>(dqkv + (long)row * D + d1) = x1;
  *reinterpret_cast<s16x8*>(dqkv + (long)row * D + d2) = x2;
}

// threads to a workgroup: a wave each where few units would leave most CUs without one (64
// rows of 2048 decoding, with the positions asked for first, 6.3 -> 5.2 us)
inline unsigned qkv_block(unsigned units) { return units <= 1u << 16 ? 64 : 256; }

// f(first token, units) for launches whose units fit 32 bits
template <typename F>
inline void by_tokens(long T, long per_token, F f) {
  const long step = std::max<long>(1, (1L << 31) / per_token);
  for (long t0 = 0; t0 < T; t0 += step) f(t0, (unsigned)(std::min(step, T - t0) * per_token));
}
