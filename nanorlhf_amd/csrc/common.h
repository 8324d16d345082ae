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
DEVINL float wave_sum(float v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
  return v;
}

DEVINL float wave_max(float v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v = fmaxf(v, __shfl_xor(v, off));
  return v;
}

// block reduction via LDS (block size multiple of 64)
template <int BLOCK>
DEVINL float block_sum(float v, float* lds_scratch /* BLOCK/64 floats */) {
  const int lane = threadIdx.x & 63;
  const int wid = threadIdx.x >> 6;
  v = wave_sum(v);
  if (lane == 0) lds_scratch[wid] = v;
  __syncthreads();
  float out = 0.f;
  if (wid == 0) {
    float x = (lane < BLOCK / 64) ? lds_scratch[lane] : 0.f;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) x += __shfl_xor(x, off);
    out = x;
    if (lane == 0) lds_scratch[0] = out;
  }
  __syncthreads();
  out = lds_scratch[0];
  __syncthreads();
  return out;
}

template <int BLOCK>
DEVINL float block_max(float v, float* lds_scratch) {
  const int lane = threadIdx.x & 63;
  const int wid = threadIdx.x >> 6;
  v = wave_max(v);
  if (lane == 0) lds_scratch[wid] = v;
  __syncthreads();
  if (wid == 0) {
    float x = (lane < BLOCK / 64) ? lds_scratch[lane] : -INFINITY;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) x = fmaxf(x, __shfl_xor(x, off));
    if (lane == 0) lds_scratch[0] = x;
  }
  __syncthreads();
  float out = lds_scratch[0];
  __syncthreads();
  return out;
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
