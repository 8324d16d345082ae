// Shared device helpers for the nanorlhf_amd gfx950 kernels.
// CDNA4: wavefront = 64 lanes, 4x SIMD-32 per CU, LDS 160 KiB/CU.
#pragma once

#include <hip/hip_runtime.h>
#include <hip/hip_bf16.h>

#define DEVINL __device__ __forceinline__

typedef __hip_bfloat16 bf16_t;

// vector types for 8/16-byte loads (guide G13: always vectorize bf16 loads)
typedef short s16x4 __attribute__((ext_vector_type(4)));   // 4 bf16 = 8 B
typedef short s16x8 __attribute__((ext_vector_type(8)));   // 8 bf16 = 16 B
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef short bf16x8_frag __attribute__((ext_vector_type(8)));  // MFMA A/B frag (4 VGPR)

DEVINL float bf2f(short x) {
  union { float f; unsigned int u; } c;
  c.u = ((unsigned int)(unsigned short)x) << 16;
  return c.f;
}

DEVINL short f2bf(float f) { return __builtin_bit_cast(short, (__bf16)f); }
// two at once; as a vector, or the compiler converts each by itself and joins them
DEVINL unsigned pack2bf(float lo, float hi) {
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(unsigned, __builtin_convertvector(f32x2{lo, hi}, bf16x2));
}

// ---- element access shared by kernels templated on bf16 (short) / float ----
DEVINL float ldf(const short* p) { return bf2f(*p); }
DEVINL float ldf(const float* p) { return *p; }
DEVINL void stf(short* p, float v) { *p = f2bf(v); }
DEVINL void stf(float* p, float v) { *p = v; }

// VEC consecutive elements as float; VEC > 1 needs VEC-element alignment
template <int VEC>
DEVINL void ldv(const float* p, float* o) {
  if constexpr (VEC % 4 == 0) {
#pragma unroll
    for (int i = 0; i < VEC; i += 4) {
      f32x4 v = *reinterpret_cast<const f32x4*>(p + i);
#pragma unroll
      for (int j = 0; j < 4; j++) o[i + j] = v[j];
    }
  } else {
#pragma unroll
    for (int i = 0; i < VEC; i++) o[i] = p[i];
  }
}
template <int VEC>
DEVINL void ldv(const short* p, float* o) {
  if constexpr (VEC == 8) {
    s16x8 v = *reinterpret_cast<const s16x8*>(p);
#pragma unroll
    for (int j = 0; j < 8; j++) o[j] = bf2f(v[j]);
  } else if constexpr (VEC == 4) {
    s16x4 v = *reinterpret_cast<const s16x4*>(p);
#pragma unroll
    for (int j = 0; j < 4; j++) o[j] = bf2f(v[j]);
  } else {
#pragma unroll
    for (int i = 0; i < VEC; i++) o[i] = bf2f(p[i]);
  }
}
template <int VEC>
DEVINL void stv(float* p, const float* v) {
  if constexpr (VEC % 4 == 0) {
#pragma unroll
    for (int i = 0; i < VEC; i += 4)
      *reinterpret_cast<f32x4*>(p + i) = f32x4{v[i], v[i + 1], v[i + 2], v[i + 3]};
  } else {
#pragma unroll
    for (int i = 0; i < VEC; i++) p[i] = v[i];
  }
}
template <int VEC>
DEVINL void stv(short* p, const float* v) {
  if constexpr (VEC == 8) {
    *reinterpret_cast<uint4*>(p) = uint4{pack2bf(v[0], v[1]), pack2bf(v[2], v[3]),
                                         pack2bf(v[4], v[5]), pack2bf(v[6], v[7])};
  } else if constexpr (VEC == 4) {
    *reinterpret_cast<uint2*>(p) = uint2{pack2bf(v[0], v[1]), pack2bf(v[2], v[3])};
  } else {
#pragma unroll
    for (int i = 0; i < VEC; i++) p[i] = f2bf(v[i]);
  }
}

// 8 elements of the sum of `splits` (at most 8) parts of a product's depth, `stride` elements
// apart, and its bias if there is one, rounded as the product's output is
DEVINL s16x8 sum_parts8(const float* p, long stride, int splits, const short* bias) {
  float v[8][8];
#pragma unroll
  for (int k = 0; k < 8; k++)
    if (k < splits) ldv<8>(p + k * stride, v[k]);
  float b[8] = {};
  if (bias) ldv<8>(bias, b);
#pragma unroll
  for (int k = 1; k < 8; k++)
    if (k < splits) {
#pragma unroll
      for (int j = 0; j < 8; j++) v[0][j] += v[k][j];
    }
  s16x8 o;
#pragma unroll
  for (int j = 0; j < 8; j++) o[j] = f2bf(v[0][j] + b[j]);
  return o;
}

// ---- activations (32-bit) -------------------------------------------------
DEVINL float act_sigmoid(float x) { return 1.f / (1.f + expf(-x)); }
DEVINL float act_silu(float x) { return x / (1.f + expf(-x)); }
DEVINL float act_gelu_tanh(float x) {
  return 0.5f * x * (1.f + tanhf(0.7978845608028654f * (x + 0.044715f * x * x * x)));
}

// ---- wave (64-lane) reductions ------------------------------------------
// All lanes get the result, exchanged between halves, rows of 16 and within a row by
// the VALU itself: through LDS (__shfl_xor), which 16 waves of a workgroup share, an
// exchange takes 107 cycles, a swap of rows 62 and a rotation in a row 27.  Pairs are
// 32, 16, 8, 4, 2 and 1 lanes apart; from 8 on every row holds the same, so that a
// rotation by 4 is that exchange too.
template <int CTRL>
DEVINL float row_move(float v) {
  return __int_as_float(
      __builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true));
}
template <typename F>
DEVINL float wave_reduce(float v, F f) {
  const auto h = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = f(__uint_as_float(h[0]), __uint_as_float(h[1]));
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = f(__uint_as_float(r[0]), __uint_as_float(r[1]));
  v = f(v, row_move<0x128>(v));     // row_ror:8
  v = f(v, row_move<0x124>(v));     // row_ror:4
  v = f(v, row_move<0x4e>(v));      // quad_perm:[2,3,0,1]
  return f(v, row_move<0xb1>(v));   // quad_perm:[1,0,3,2]
}
DEVINL float wave_sum(float v) { return wave_reduce(v, [](float a, float b) { return a + b; }); }
DEVINL float wave_max(float v) { return wave_reduce(v, [](float a, float b) { return fmaxf(a, b); }); }

// block reduction via LDS (block size a multiple of 64, up to 1024): every thread reduces
// the waves' results, in pairs of 8, 4, 2 and 1 waves apart.  1024 threads: 2700 cycles
// with exchanges through LDS and the first wave reducing for all.
template <int BLOCK, typename F>
DEVINL float block_reduce(float v, float* lds_scratch /* BLOCK/64 floats */, F f) {
  constexpr int W = BLOCK / 64;
  static_assert((W & (W - 1)) == 0 && W <= 16, "a power of two of waves");
  v = wave_reduce(v, f);
  if constexpr (W == 1) return v;
  if ((threadIdx.x & 63) == 0) lds_scratch[threadIdx.x >> 6] = v;
  __syncthreads();
  float x[W];
#pragma unroll
  for (int w = 0; w < W; w++) x[w] = lds_scratch[w];
#pragma unroll
  for (int off = W / 2; off > 0; off >>= 1)
#pragma unroll
    for (int w = 0; w < off; w++) x[w] = f(x[w], x[w + off]);
  __syncthreads();
  return x[0];
}
template <int BLOCK>
DEVINL float block_sum(float v, float* lds_scratch) {
  return block_reduce<BLOCK>(v, lds_scratch, [](float a, float b) { return a + b; });
}
template <int BLOCK>
DEVINL float block_max(float v, float* lds_scratch) {
  return block_reduce<BLOCK>(v, lds_scratch, [](float a, float b) { return fmaxf(a, b); });
}

// ---- counter-based RNG (deterministic replay) ----------------------------
DEVINL unsigned long long splitmix64(unsigned long long x) {
  x += 0x9E3779B97F4A7C15ull;
  x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
  x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
  return x ^ (x >> 31);
}

DEVINL float hash_uniform(unsigned long long seed, unsigned long long step,
                          unsigned long long row) {
  unsigned long long h = splitmix64(seed ^ splitmix64(step ^ splitmix64(row)));
  // top 24 bits -> [0,1)
  return (float)(h >> 40) * (1.0f / 16777216.0f);
}

// ---- bf16 matrix cores on 32-bit values: x = hi + lo, both bf16 -------------
typedef __bf16 bf16x8l __attribute__((ext_vector_type(8)));

DEVINL f32x4 mfma16l(bf16x8l a, bf16x8l b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
DEVINL bf16x8l frag(const short* p) { return *reinterpret_cast<const bf16x8l*>(p); }
DEVINL float silu_fast(float x) { return x * __builtin_amdgcn_rcpf(1.f + __expf(-x)); }

DEVINL void split4(const float* x, s16x4& hi, s16x4& lo) {
#pragma unroll
  for (int j = 0; j < 4; j++) {
    hi[j] = f2bf(x[j]);
    lo[j] = f2bf(x[j] - bf2f(hi[j]));
  }
}
DEVINL void split8(const float* x, s16x8& hi, s16x8& lo) {
#pragma unroll
  for (int j = 0; j < 8; j++) {
    hi[j] = f2bf(x[j]);
    lo[j] = f2bf(x[j] - bf2f(hi[j]));
  }
}
DEVINL bf16x8l as_frag(const s16x8& x) { return *reinterpret_cast<const bf16x8l*>(&x); }

// 16 (or 4) bytes per lane from base + offset to LDS, lane after lane from `at`;
// base and at are the same in the whole wave.  As assembly, because the compiler
// waits for a load that it knows to write LDS before the next LDS read, whichever
// buffer that reads, and so undoes a prefetch; there is no output register, and
// nothing else on this part uses m0.  The caller waits (wait_loads).
DEVINL const void* in_sgprs(const void* p) {
  const unsigned long long x = (unsigned long long)p;
  return (const void*)((unsigned long long)__builtin_amdgcn_readfirstlane((unsigned)(x >> 32)) << 32 |
                       (unsigned)__builtin_amdgcn_readfirstlane((unsigned)x));
}
DEVINL unsigned lds_address(const void* p) {
  return __builtin_amdgcn_readfirstlane(
      (unsigned)(size_t)(const __attribute__((address_space(3))) void*)p);
}
DEVINL void load_to_lds16(const void* base, unsigned offset, const void* at) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
               ::"s"(lds_address(at)), "v"(offset), "s"(in_sgprs(base)) : "memory");
}
// the same with an address for every lane
DEVINL void load_to_lds16(const void* p, const void* at) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off"
               ::"s"(lds_address(at)), "v"(p) : "memory");
}
DEVINL void load_to_lds4(const void* base, unsigned offset, const void* at) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2"
               ::"s"(lds_address(at)), "v"(offset), "s"(in_sgprs(base)) : "memory");
}

// until at most N loads of this wave are outstanding
template <int N>
DEVINL void wait_loads() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt((N & 15) | (N >> 4) << 14 | 0x0f70);   // vmcnt alone
  asm volatile("" ::: "memory");
}

// The oldest of a ring of R chunks, L loads of this wave each, has arrived, if at
// most `left` younger ones are under way.
template <int L, int R>
DEVINL void chunk_ready(int left) {
  static_assert(R <= 4 && L * (R - 1) < 64, "vmcnt");
  if (left >= R - 1) wait_loads<L * (R - 1)>();
  else if (R > 3 && left == 2) wait_loads<L * 2>();
  else if (R > 2 && left == 1) wait_loads<L>();
  else wait_loads<0>();
}

// wave-private LDS write->read ordering (staging buffers written and read
// by the same wave between barriers)
DEVINL void lds_fence_wave_kv() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

#define HIP_CHECK_LAST()                                                    \
  do {                                                                      \
    hipError_t e_ = hipGetLastError();                                      \
    if (e_ != hipSuccess) {                                                 \
      TORCH_CHECK(false, "HIP kernel launch failed: ", hipGetErrorString(e_)); \
    }                                                                       \
  } while (0)
