// Row-major bf16 tiles of TILE rows in LDS, filled by direct loads and read as
// fragments of 32x32x16 products along either dimension.
#pragma once

#include <hip/hip_runtime.h>

#include "common.h"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));

DEVINL f32x16_t mfma32x32x16(bf16x8 a, bf16x8 b, f32x16_t c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

constexpr int TILE = 64;     // rows of a tile

// row of register r of a 32x32 result in lane half `hi`
DEVINL int crow(int r, int hi) { return (r & 3) + 8 * (r >> 2) + 4 * hi; }

// [row][D] bf16, 16-byte chunks exchanged (xor) by row:
// 16 rows x one chunk (a fragment read along D) and 4 rows x 4 chunks (half a
// transposed read) both have to touch all 64 banks once.  Rows 256 bytes apart
// start at the same bank, so the row's low two bits move a chunk between the
// groups of four that a transposed read takes, the next two within a group.
template <int D>
DEVINL int swz(int row) {
  if constexpr (D == 128) return ((row & 3) << 2) | ((row >> 2) & 3);
  else if constexpr (D == 64) return (((row >> 1) & 1) << 2) | ((row >> 2) & 3);
  else return (row >> 2) & 3;
}

// All waves' loads into LDS have arrived, and nobody reads the buffer that is
// filled next.
DEVINL void tiles_ready() {
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
}

// the TILE rows from src on (row stride `ld` elements; rows from `left` on
// repeat the last) into a tile; a lane fetches the chunk that its 16 bytes of
// the tile hold
template <int D>
DEVINL void stage_tile(const short* src, int ld, int left, const short* tile) {
  constexpr int SLOTS = TILE * D / 8;
  const int wave0 = __builtin_amdgcn_readfirstlane(threadIdx.x) & ~63;
#pragma unroll
  for (int i = 0; i < SLOTS; i += 256) {
    const int idx = i + threadIdx.x;
    const int row = idx / (D / 8), c = (idx % (D / 8)) ^ swz<D>(row);
    load_to_lds16(src, (unsigned)(min(row, left - 1) * ld + c * 8) * 2, tile + (i + wave0) * 8);
  }
}

// 8 consecutive d (from 16 * ds + 8 * half) of row r0 + lane % 32
template <int D>
DEVINL bf16x8 row_frag(const short* tile, int r0, int ds, int lane) {
  const int row = r0 + (lane & 31);
  return *reinterpret_cast<const bf16x8*>(
      tile + row * D + (((2 * ds + (lane >> 5)) ^ swz<D>(row)) << 3));
}

// column d0 + lane % 32, rows r0 + {0-3, 8-11} + 4 * half, the order of a result's
// registers, or (IN_ORDER) r0 + 8 * half + {0-7}, that of row_frag (r0 a multiple of 16)
template <int D, bool IN_ORDER = false>
DEVINL bf16x8 col_frag(const short* tile, int r0, int d0, int lane) {
  typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
  const int i = lane & 15;
  const int col = d0 + (lane & 16) + (i & 3) * 4;
  union { s16x4 h[2]; bf16x8 f; } u;
#pragma unroll
  for (int p = 0; p < 2; p++) {
    const int row = r0 + (IN_ORDER ? 4 : 8) * p + (IN_ORDER ? 8 : 4) * (lane >> 5) + (i >> 2);
    const short* a = tile + row * D + (((col >> 3) ^ swz<D>(row)) << 3) + (col & 7);
    u.h[p] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)a);
  }
  return u.f;
}

// The same fragments from an address that all of a tile share: with `at` = the tile's
// byte address + row_at<D>(lane) or col_at<D>(lane), another ds (or 32 columns) is an
// xor of a constant, another 32 (16) rows an offset.  One register instead of one per
// fragment.
template <int D>
DEVINL unsigned row_at(int lane) {
  const int row = lane & 31;
  return row * 2 * D + (((lane >> 5) ^ swz<D>(row)) << 4);
}
template <int D>
DEVINL unsigned col_at(int lane) {
  const int i = lane & 15, col = (lane & 16) + (i & 3) * 4;
  const int row = 4 * (lane >> 5) + (i >> 2);
  return row * 2 * D + (((col >> 3) ^ swz<D>(row)) << 4) + (col & 7) * 2;
}
template <int D>
DEVINL bf16x8 row_frag_at(unsigned at, int r0, int ds) {
  typedef __attribute__((address_space(3))) const char* lds_bytes;
  typedef __attribute__((address_space(3))) const bf16x8* lds_frag;
  return *(lds_frag)((lds_bytes)(at ^ ds << 5) + r0 * 2 * D);
}
template <int D>
DEVINL bf16x8 col_frag_at(unsigned at, int r0, int d0) {
  typedef __attribute__((address_space(3))) char* lds_bytes;
  typedef __attribute__((address_space(3))) s16x4* lds_s16x4;
  union { s16x4 h[2]; bf16x8 f; } u;
#pragma unroll
  for (int p = 0; p < 2; p++)       // 8 rows on, the swizzle has its second bit changed
    u.h[p] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (lds_s16x4)((lds_bytes)(at ^ (d0 << 1 | p << 5)) + (r0 + 8 * p) * 2 * D));
  return u.f;
}
