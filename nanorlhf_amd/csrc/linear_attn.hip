// Linear attention with one fixed decay per head and no denominator:
//   S_t = decay S_(t-1) + k_t v_t^T,   o_t = S_t^T q_t,   S [D, V] in 32-bit.
// q, k, v are read from columns of a projection row; on the way in they pass
// an optional SiLU, an optional rotation of the first dims (k also a factor).
//
// Portions of prompts run in chunks of 64 tokens (never across sequences):
//   1. chunk_state: what each chunk adds to the state, in parallel;
//   2. chunk_scan:  a running state over each sequence's chunks, from the
//                   sequence's slot (or zero) and back into it;
//   3. chunk_out:   decayed (q k^T) v inside a chunk plus q times the state
//                   ahead of it, in parallel.
// bf16 rows that can be read four elements at a time, of heads up to 128 wide, run the same by
// segments of several chunks (below).
// Products run on the matrix cores.  float32 inputs use float32 MFMA.  bf16
// inputs use bf16 MFMA on split operands: whatever is 32-bit (rotated and
// decayed q and k, decayed scores, the state) is the sum of two bf16 numbers,
// hi + lo, and a product is the sum of the significant cross terms, so about
// 16 bits of every operand count; v is bf16 as the projection left it.
//
// Single tokens (decode) update the state in place: one workgroup per
// (sequence, head) streams S once through registers.
#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>

#include <algorithm>

#include "common.h"
#include "checks.h"

constexpr int CHUNK = 64;
constexpr int VBLK = 64;

DEVINL f32x4 mfma4f(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// where q/k/v come from and what happens to them on the way in
struct Source {
  long ld;                 // projection row stride
  int H, D, V;
  const float* cs;         // [T, rdims] cos | sin, or null
  int rdims, interleaved, silu;
  float kscale;
};

struct Chunks {
  const int* seq;          // [n] sequence of a chunk
  const int* row;          // [n] its first token row
  const int* len;          // [n] its tokens, 1..CHUNK
  const int* first;        // [B + 1] first chunk of a sequence
};

template <typename T>
DEVINL float load_qk(const T* base, int e, const Source& s, const float* cs) {
  float x = ldf(base + e);
  if (s.silu) x = act_silu(x);
  if (e < s.rdims) {
    const int half = s.rdims >> 1;
    const int p = s.interleaved ? e >> 1 : (e < half ? e : e - half);
    const bool lead = s.interleaved ? !(e & 1) : e < half;
    const int other = s.interleaved ? e ^ 1 : (lead ? e + half : e - half);
    float y = ldf(base + other);
    if (s.silu) y = act_silu(y);
    x = x * cs[p] + (lead ? -y : y) * cs[half + p];
  }
  return x;
}

template <typename T>
DEVINL float load_v(const T* base, int e, const Source& s) {
  const float x = ldf(base + e);
  return s.silu ? act_silu(x) : x;
}

// ------------------------------------------------ 1. what a chunk adds
// U[d][v] = sum_j decay^(n-1-j) k_j[d] v_j[v]; ws [chunks, H, D, V]
template <typename T, int DP>
__global__ __launch_bounds__(256) void chunk_state_kernel(
    const T* __restrict__ k, const T* __restrict__ v, Source s, Chunks ch,
    const float* __restrict__ pw, float* __restrict__ ws) {
  constexpr int KS = DP + 16, VS = VBLK + 16;
  __shared__ float kt[CHUNK * KS], vt[CHUNK * VS];
  const int c = blockIdx.x, h = blockIdx.y, v0 = blockIdx.z * VBLK;
  const int n = ch.len[c];
  const long t0 = ch.row[c];
  const float* pwh = pw + h * (CHUNK + 1);
  for (int i = threadIdx.x; i < CHUNK * DP; i += 256) {
    const int j = i / DP, d = i % DP;
    float x = 0.f;
    if (j < n && d < s.D)
      x = load_qk(k + (t0 + j) * s.ld + h * s.D, d, s, s.cs + (t0 + j) * s.rdims) * s.kscale *
          pwh[n - 1 - j];
    kt[j * KS + d] = x;
  }
  for (int i = threadIdx.x; i < CHUNK * VBLK; i += 256) {
    const int j = i / VBLK, e = i % VBLK;
    vt[j * VS + e] =
        (j < n && v0 + e < s.V) ? load_v(v + (t0 + j) * s.ld + h * s.V, v0 + e, s) : 0.f;
  }
  __syncthreads();
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int lo = lane & 15, hi = lane >> 4;
  constexpr int RT = DP / 16;                 // row tiles of U
  constexpr int RW = RT >= 4 ? RT / 4 : RT;   // per wave
  constexpr int CW = RT >= 4 ? 4 : 1;         // column tiles per wave
  const int r0 = RT >= 4 ? w * RW : 0, c0 = RT >= 4 ? 0 : w;
  f32x4 acc[RW][CW];
#pragma unroll
  for (int r = 0; r < RW; r++)
#pragma unroll
    for (int q = 0; q < CW; q++) acc[r][q] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int st = 0; st < CHUNK / 4; st++) {
    const int j = 4 * st + hi;
    float a[RW], b[CW];
#pragma unroll
    for (int r = 0; r < RW; r++) a[r] = kt[j * KS + (r0 + r) * 16 + lo];
#pragma unroll
    for (int q = 0; q < CW; q++) b[q] = vt[j * VS + (c0 + q) * 16 + lo];
#pragma unroll
    for (int r = 0; r < RW; r++)
#pragma unroll
      for (int q = 0; q < CW; q++) acc[r][q] = mfma4f(a[r], b[q], acc[r][q]);
  }
  float* u = ws + ((long)c * s.H + h) * s.D * s.V;
#pragma unroll
  for (int r = 0; r < RW; r++)
#pragma unroll
    for (int q = 0; q < CW; q++)
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const int d = (r0 + r) * 16 + 4 * hi + i, e = v0 + (c0 + q) * 16 + lo;
        if (d < s.D && e < s.V) u[(long)d * s.V + e] = acc[r][q][i];
      }
}

// ------------------------------------------------------ 2. running state
// ws: in, what a chunk adds; out, the state ahead of the chunk
__global__ __launch_bounds__(256) void chunk_scan_kernel(
    float* __restrict__ ws, float* __restrict__ state, Chunks ch,
    const int* __restrict__ slots, const int* __restrict__ fresh,
    const float* __restrict__ pw, int H, int DV) {
  const int b = blockIdx.x, h = blockIdx.y;
  const int e = blockIdx.z * 256 + threadIdx.x;
  if (e >= DV) return;
  float* st = state + ((long)slots[b] * H + h) * DV + e;
  const float* pwh = pw + h * (CHUNK + 1);
  float s = fresh[b] ? 0.f : *st;
  const int c1 = ch.first[b + 1];
  float* p = ws + ((long)ch.first[b] * H + h) * DV + e;
#pragma unroll 4
  for (int c = ch.first[b]; c < c1; c++, p += (long)H * DV) {
    const float u = *p;
    *p = s;
    s = pwh[ch.len[c]] * s + u;
  }
  *st = s;
}

// ---------------------------------------------------------- 3. the output
template <typename T, int DP>
__global__ __launch_bounds__(256) void chunk_out_kernel(
    const T* __restrict__ q, const T* __restrict__ k, const T* __restrict__ v, Source s,
    Chunks ch, const float* __restrict__ pw, const float* __restrict__ ws, T* __restrict__ o, long ldo) {
  constexpr int KS = DP + 4, VS = VBLK + 16, PS = CHUNK + 4;
  __shared__ float kt[CHUNK * KS], vt[CHUNK * VS], pt[4][16 * PS], pws[CHUNK + 1];
  const int c = blockIdx.x, h = blockIdx.y, v0 = blockIdx.z * VBLK;
  const int n = ch.len[c];
  const long t0 = ch.row[c];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int lo = lane & 15, hi = lane >> 4;
  if (threadIdx.x <= CHUNK) pws[threadIdx.x] = pw[h * (CHUNK + 1) + threadIdx.x];
  auto stage = [&](const T* x, float mul) {
    for (int i = threadIdx.x; i < CHUNK * DP; i += 256) {
      const int j = i / DP, d = i % DP;
      kt[j * KS + d] = (j < n && d < s.D) ? load_qk(x + (t0 + j) * s.ld + h * s.D, d, s,
                                                    s.cs + (t0 + j) * s.rdims) * mul
                                          : 0.f;
    }
  };
  stage(q, 1.f);
  __syncthreads();
  float qf[DP / 4];
#pragma unroll
  for (int st = 0; st < DP / 4; st++) qf[st] = kt[(16 * w + lo) * KS + 4 * st + hi];
  __syncthreads();
  stage(k, s.kscale);
  for (int i = threadIdx.x; i < CHUNK * VBLK; i += 256) {
    const int j = i / VBLK, e = i % VBLK;
    vt[j * VS + e] =
        (j < n && v0 + e < s.V) ? load_v(v + (t0 + j) * s.ld + h * s.V, v0 + e, s) : 0.f;
  }
  __syncthreads();
  if (16 * w >= n) return;
  f32x4 acc[4];
#pragma unroll
  for (int t = 0; t < 4; t++) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  // q decayed to the chunk's start, times the state ahead of the chunk
  const float* sp = ws + ((long)c * s.H + h) * s.D * s.V;
  const float pq = pws[16 * w + lo + 1];
#pragma unroll 4
  for (int st = 0; st < DP / 4; st++) {
    const int d = 4 * st + hi;
    const float a = qf[st] * pq;
#pragma unroll
    for (int t = 0; t < 4; t++) {
      const int e = v0 + 16 * t + lo;
      const float b = (d < s.D && e < s.V) ? sp[(long)d * s.V + e] : 0.f;
      acc[t] = mfma4f(a, b, acc[t]);
    }
  }
  // inside the chunk
  float* pr = pt[w];
  for (int jt = 0; jt <= w; jt++) {
    f32x4 sc{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int st = 0; st < DP / 4; st++)
      sc = mfma4f(qf[st], kt[(16 * jt + lo) * KS + 4 * st + hi], sc);
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int i = 16 * w + 4 * hi + r, j = 16 * jt + lo;
      pr[(4 * hi + r) * PS + j] = i >= j ? sc[r] * pws[i - j] : 0.f;
    }
  }
  lds_fence_wave_kv();
  for (int st = 0; st < 4 * (w + 1); st++) {
    const float a = pr[lo * PS + 4 * st + hi];
#pragma unroll
    for (int t = 0; t < 4; t++)
      acc[t] = mfma4f(a, vt[(4 * st + hi) * VS + 16 * t + lo], acc[t]);
  }
#pragma unroll
  for (int t = 0; t < 4; t++)
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int i = 16 * w + 4 * hi + r, e = v0 + 16 * t + lo;
      if (i < n && e < s.V) stf(o + (t0 + i) * ldo + h * s.V + e, acc[t][r]);
    }
}

// ===================================================== bf16: split operands
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

// SiLU and rotation of two runs that hold whole pairs
DEVINL void shape_runs(float* a, float* b, const Source& s, bool rot, const float* c,
                       const float* sn) {
  if (s.silu) {
#pragma unroll
    for (int j = 0; j < 4; j++) {
      a[j] = silu_fast(a[j]);
      b[j] = silu_fast(b[j]);
    }
  }
  if (!rot) return;
  if (s.interleaved) {
#pragma unroll
    for (int j = 0; j < 4; j += 2) {
      const float u = a[j], v = a[j + 1];
      a[j] = u * c[j / 2] - v * sn[j / 2];
      a[j + 1] = v * c[j / 2] + u * sn[j / 2];
      const float x = b[j], y = b[j + 1];
      b[j] = x * c[2 + j / 2] - y * sn[2 + j / 2];
      b[j + 1] = y * c[2 + j / 2] + x * sn[2 + j / 2];
    }
  } else {
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const float u = a[j], v = b[j];
      a[j] = u * c[j] - v * sn[j];
      b[j] = v * c[j] + u * sn[j];
    }
  }
}

// Eight elements of one q or k row, as two runs of four: a at element ea, b at
// eb.  Run g holds whole rotation pairs (with `vec`; without it, elements 8g..
// 8g+7 one by one).  Elements past D are 0.
DEVINL void load_runs(const short* row, int g, const Source& s, const float* cs, bool vec,
                      float* a, float* b, int& ea, int& eb) {
  if (!vec) {
    ea = 8 * g;
    eb = ea + 4;
#pragma unroll
    for (int j = 0; j < 4; j++) {
      a[j] = ea + j < s.D ? load_qk(row, ea + j, s, cs) : 0.f;
      b[j] = eb + j < s.D ? load_qk(row, eb + j, s, cs) : 0.f;
    }
    return;
  }
  const int half = s.rdims >> 1, p = 4 * g;      // first of four pairs
  const bool rot = p < half;
  if (s.interleaved || !rot) {
    ea = rot || s.interleaved ? 2 * p : s.rdims + 2 * (p - half);
    eb = ea + 4;
  } else {
    ea = p;
    eb = half + p;
  }
#pragma unroll
  for (int j = 0; j < 4; j++) a[j] = b[j] = 0.f;
  if (ea < s.D) ldv<4>(row + ea, a);
  if (eb < s.D) ldv<4>(row + eb, b);
  float c[4], sn[4];
  if (rot) {
    ldv<4>(cs + p, c);
    ldv<4>(cs + half + p, sn);
  }
  shape_runs(a, b, s, rot, c, sn);
}

constexpr int TS = CHUNK + 8;    // LDS row of a [feature][token] tile

// Four tokens by four columns of v, turned around for a tile vt[e][j] =
// v_j[v0 + e]; 0 past the chunk's tokens and past V.
template <int VB>
struct VPatch {
  static constexpr int COUNT = (CHUNK / 4) * (VB / 4);
  s16x4 col[4];
  int e, j;
  DEVINL void load(int i, const short* v, const Source& s, long t0, int n, int h, int v0,
                   bool vec) {
    e = (i % (VB / 4)) * 4;
    j = (i / (VB / 4)) * 4;
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const short* row = v + (t0 + j + r) * s.ld + h * s.V + v0 + e;
      float x[4] = {0.f, 0.f, 0.f, 0.f};
      if (j + r < n) {
        if (vec) {
          if (v0 + e < s.V) ldv<4>(row, x);
        } else {
#pragma unroll
          for (int c = 0; c < 4; c++)
            if (v0 + e + c < s.V) x[c] = ldf(row + c);
        }
      }
#pragma unroll
      for (int c = 0; c < 4; c++) col[c][r] = f2bf(s.silu ? silu_fast(x[c]) : x[c]);
    }
  }
  DEVINL void store(short* vt) const {
#pragma unroll
    for (int c = 0; c < 4; c++) *reinterpret_cast<s16x4*>(vt + (e + c) * TS + j) = col[c];
  }
};

// ws [chunks, H, V, DP]: what a chunk adds, feature-major
template <int DP, int VB>
__global__ __launch_bounds__(512) void chunk_state_split_kernel(
    const short* __restrict__ k, const short* __restrict__ v, Source s, Chunks ch,
    const float* __restrict__ pw, float* __restrict__ ws, bool vec) {
  __shared__ __attribute__((aligned(16))) short kt[2][DP * TS], vt[VB * TS];
  const int c = blockIdx.x, h = blockIdx.y, v0 = blockIdx.z * VB;
  const int n = ch.len[c];
  const long t0 = ch.row[c];
  const float* pwh = pw + h * (CHUNK + 1);
  // one half of the workgroup stages v, the other k
  if (threadIdx.x >= 256) {
    for (int i = threadIdx.x - 256; i < VPatch<VB>::COUNT; i += 256) {
      VPatch<VB> x;
      x.load(i, v, s, t0, n, h, v0, vec);
      x.store(vt);
    }
  } else for (int i = threadIdx.x; i < (CHUNK / 4) * (DP / 8); i += 256) {
    const int g = i % (DP / 8), j = (i / (DP / 8)) * 4;
    float a[4][4], b[4][4];
    int ea = 8 * g, eb = ea + 4;
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const bool live = j + r < n;
      const long t = t0 + (live ? j + r : 0);
      load_runs(k + t * s.ld + h * s.D, g, s, s.cs + t * s.rdims, vec, a[r], b[r], ea, eb);
      const float m = live ? s.kscale * pwh[n - 1 - j - r] : 0.f;
#pragma unroll
      for (int q = 0; q < 4; q++) {
        a[r][q] *= m;
        b[r][q] *= m;
      }
    }
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const float x[4] = {a[0][q], a[1][q], a[2][q], a[3][q]};
      const float y[4] = {b[0][q], b[1][q], b[2][q], b[3][q]};
      s16x4 hi, lo;
      split4(x, hi, lo);
      *reinterpret_cast<s16x4*>(&kt[0][(ea + q) * TS + j]) = hi;
      *reinterpret_cast<s16x4*>(&kt[1][(ea + q) * TS + j]) = lo;
      split4(y, hi, lo);
      *reinterpret_cast<s16x4*>(&kt[0][(eb + q) * TS + j]) = hi;
      *reinterpret_cast<s16x4*>(&kt[1][(eb + q) * TS + j]) = lo;
    }
  }
  __syncthreads();
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int lo = lane & 15, hi = lane >> 4;
  constexpr int CT = VB / 16;                  // v tiles: 4 or 8
  constexpr int RW = DP / 16 * CT / 8;         // feature tiles per wave
  const int ct = w % CT, r0 = (w / CT) * RW;
  bf16x8l vf[2];
#pragma unroll
  for (int ks = 0; ks < 2; ks++) vf[ks] = frag(&vt[(ct * 16 + lo) * TS + 32 * ks + 8 * hi]);
  const int e = v0 + ct * 16 + lo;
  float* u = ws + (((long)c * s.H + h) * s.V + e) * DP;
#pragma unroll 4
  for (int rt = r0; rt < r0 + RW; rt++) {
    f32x4 acc{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < 2; ks++) {
      const int at = (16 * rt + lo) * TS + 32 * ks + 8 * hi;
      acc = mfma16l(frag(&kt[1][at]), vf[ks], acc);
      acc = mfma16l(frag(&kt[0][at]), vf[ks], acc);
    }
    if (e < s.V) *reinterpret_cast<f32x4*>(u + 16 * rt + 4 * hi) = acc;
  }
}

// in place: what a chunk adds -> the state ahead of it, as hi | lo << 16.
// The slot itself is exchanged in full float32, [D][V].
__global__ __launch_bounds__(256) void chunk_scan_split_kernel(
    float* __restrict__ ws, float* __restrict__ state, Chunks ch,
    const int* __restrict__ slots, const int* __restrict__ fresh,
    const float* __restrict__ pw, int H, int D, int V, int DP) {
  constexpr int AHEAD = 8;
  const int b = blockIdx.x, h = blockIdx.y;
  const int e = blockIdx.z * 256 + threadIdx.x;
  if (e >= V * DP) return;
  const int vi = e / DP, d = e % DP;
  const bool real = d < D;
  float* st = state + (((long)slots[b] * H + h) * D + (real ? d : 0)) * V + vi;
  const float* pwh = pw + h * (CHUNK + 1);
  float s = (fresh[b] || !real) ? 0.f : *st;
  const int c0 = ch.first[b], c1 = ch.first[b + 1];
  const long step = (long)H * V * DP;
  float* p = ws + ((long)c0 * H + h) * V * DP + e;
  for (int c = c0; c < c1; c += AHEAD) {
    float u[AHEAD];
#pragma unroll
    for (int i = 0; i < AHEAD; i++) u[i] = c + i < c1 ? p[i * step] : 0.f;
#pragma unroll
    for (int i = 0; i < AHEAD; i++) {
      if (c + i >= c1) break;
      const short hi = f2bf(s), lo = f2bf(s - bf2f(hi));
      reinterpret_cast<unsigned*>(p)[i * step] =
          (unsigned)(unsigned short)hi | ((unsigned)(unsigned short)lo << 16);
      s = pwh[ch.len[c + i]] * s + u[i];
    }
    p += AHEAD * step;
  }
  if (real) *st = s;
}

// One workgroup: one chunk, one head, VB columns of v.  Everything is computed
// transposed (a lane holds one token's consecutive columns).  With a gate (V
// <= VB), the head's output leaves normed and gated.
template <int DP, int VB>
__global__ __launch_bounds__(512, DP > 128 ? 2 : 4) void chunk_out_split_kernel(
    const short* __restrict__ q, const short* __restrict__ k, const short* __restrict__ v,
    Source s, Chunks ch, const float* __restrict__ pw, const unsigned* __restrict__ ws,
    const short* __restrict__ gate, long ldg, float eps, short* __restrict__ o, long ldo,
    bool vec) {
  constexpr int QS = DP + 8;
  constexpr int PV = 2 * CHUNK * TS + VB * TS;
  constexpr int KR = 2 * CHUNK * QS > PV ? 2 * CHUNK * QS : PV;
  constexpr int CT = VB / 16;             // v tiles: 4 or 8
  constexpr int RW = CT / 2;              // token tiles per wave
  __shared__ __attribute__((aligned(16))) short qt[2][CHUNK * QS], kreg[KR];
  __shared__ float pws[CHUNK + 1], red[CT][CHUNK];
  short* kt[2] = {kreg, kreg + CHUNK * QS};
  short* pt[2] = {kreg, kreg + CHUNK * TS};    // scores and v take the keys' place
  short* vt = kreg + 2 * CHUNK * TS;
  const int c = blockIdx.x, h = blockIdx.y, v0 = blockIdx.z * VB;
  const int n = ch.len[c];
  const long t0 = ch.row[c];
  if (threadIdx.x <= CHUNK) pws[threadIdx.x] = pw[h * (CHUNK + 1) + threadIdx.x];
  for (int i = threadIdx.x; i < CHUNK * (DP / 8); i += 512) {
    const int g = i % (DP / 8), j = i / (DP / 8);
    const long t = t0 + (j < n ? j : 0);
    float a[4], b[4];
    int ea, eb;
    s16x4 hi, lo;
    load_runs(q + t * s.ld + h * s.D, g, s, s.cs + t * s.rdims, vec, a, b, ea, eb);
    split4(a, hi, lo);
    *reinterpret_cast<s16x4*>(&qt[0][j * QS + ea]) = hi;
    *reinterpret_cast<s16x4*>(&qt[1][j * QS + ea]) = lo;
    split4(b, hi, lo);
    *reinterpret_cast<s16x4*>(&qt[0][j * QS + eb]) = hi;
    *reinterpret_cast<s16x4*>(&qt[1][j * QS + eb]) = lo;
    load_runs(k + t * s.ld + h * s.D, g, s, s.cs + t * s.rdims, vec, a, b, ea, eb);
#pragma unroll
    for (int r = 0; r < 4; r++) {
      a[r] *= s.kscale;
      b[r] *= s.kscale;
    }
    split4(a, hi, lo);
    *reinterpret_cast<s16x4*>(&kt[0][j * QS + ea]) = hi;
    *reinterpret_cast<s16x4*>(&kt[1][j * QS + ea]) = lo;
    split4(b, hi, lo);
    *reinterpret_cast<s16x4*>(&kt[0][j * QS + eb]) = hi;
    *reinterpret_cast<s16x4*>(&kt[1][j * QS + eb]) = lo;
  }
  VPatch<VB> vp;
  if (threadIdx.x < VPatch<VB>::COUNT) vp.load(threadIdx.x, v, s, t0, n, h, v0, vec);
  __syncthreads();

  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int lo = lane & 15, hi = lane >> 4;
  const int ct = w % CT, r0 = (w / CT) * RW;
  const int e0 = v0 + 16 * ct;
  f32x4 acc[RW];
#pragma unroll
  for (int r = 0; r < RW; r++) acc[r] = f32x4{0.f, 0.f, 0.f, 0.f};
  // state ahead of the chunk, times q
  const unsigned* sp = ws + (((long)c * s.H + h) * s.V + min(e0 + lo, s.V - 1)) * DP;
#pragma unroll 4
  for (int ks = 0; ks < DP / 32; ks++) {
    u32x4 x = *reinterpret_cast<const u32x4*>(sp + 32 * ks + 8 * hi);
    u32x4 y = *reinterpret_cast<const u32x4*>(sp + 32 * ks + 8 * hi + 4);
    if (e0 + lo >= s.V) x = y = u32x4{0u, 0u, 0u, 0u};
    union { unsigned u[4]; bf16x8l f; } sh, sl;
    sh.u[0] = __builtin_amdgcn_perm(x[1], x[0], 0x05040100);
    sh.u[1] = __builtin_amdgcn_perm(x[3], x[2], 0x05040100);
    sh.u[2] = __builtin_amdgcn_perm(y[1], y[0], 0x05040100);
    sh.u[3] = __builtin_amdgcn_perm(y[3], y[2], 0x05040100);
    sl.u[0] = __builtin_amdgcn_perm(x[1], x[0], 0x07060302);
    sl.u[1] = __builtin_amdgcn_perm(x[3], x[2], 0x07060302);
    sl.u[2] = __builtin_amdgcn_perm(y[1], y[0], 0x07060302);
    sl.u[3] = __builtin_amdgcn_perm(y[3], y[2], 0x07060302);
#pragma unroll
    for (int r = 0; r < RW; r++) {
      const int at = (16 * (r0 + r) + lo) * QS + 32 * ks + 8 * hi;
      const bf16x8l qh = frag(&qt[0][at]), ql = frag(&qt[1][at]);
      acc[r] = mfma16l(sl.f, qh, acc[r]);
      acc[r] = mfma16l(sh.f, ql, acc[r]);
      acc[r] = mfma16l(sh.f, qh, acc[r]);
    }
  }
#pragma unroll
  for (int r = 0; r < RW; r++) acc[r] *= pws[16 * (r0 + r) + lo + 1];
  // scores of this wave's two tiles (token tile it, key tiles jt, jt + 1)
  const int it = w >> 1, jt = (w & 1) * 2;
  f32x4 sc[2];
#pragma unroll
  for (int x = 0; x < 2; x++) {
    sc[x] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (jt + x > it) continue;
#pragma unroll 4
    for (int ks = 0; ks < DP / 32; ks++) {
      const int qa = (16 * it + lo) * QS + 32 * ks + 8 * hi;
      const int ka = (16 * (jt + x) + lo) * QS + 32 * ks + 8 * hi;
      const bf16x8l qh = frag(&qt[0][qa]), ql = frag(&qt[1][qa]);
      const bf16x8l kh = frag(&kt[0][ka]), kl = frag(&kt[1][ka]);
      sc[x] = mfma16l(kl, qh, sc[x]);
      sc[x] = mfma16l(kh, ql, sc[x]);
      sc[x] = mfma16l(kh, qh, sc[x]);
    }
  }
  __syncthreads();                 // every wave is done with the keys
  if (threadIdx.x < VPatch<VB>::COUNT) vp.store(vt);
#pragma unroll
  for (int x = 0; x < 2; x++) {
    const int i = 16 * it + lo, j = 16 * (jt + x) + 4 * hi;
    float p[4];
#pragma unroll
    for (int r = 0; r < 4; r++) p[r] = i >= j + r ? sc[x][r] * pws[max(i - j - r, 0)] : 0.f;
    s16x4 ph, pl;
    split4(p, ph, pl);
    *reinterpret_cast<s16x4*>(&pt[0][i * TS + j]) = ph;
    *reinterpret_cast<s16x4*>(&pt[1][i * TS + j]) = pl;
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < RW; r++)
    for (int ks = 0; ks <= (r0 + r) / 2; ks++) {
      const bf16x8l vf = frag(&vt[(16 * ct + lo) * TS + 32 * ks + 8 * hi]);
      const int at = (16 * (r0 + r) + lo) * TS + 32 * ks + 8 * hi;
      acc[r] = mfma16l(vf, frag(&pt[1][at]), acc[r]);
      acc[r] = mfma16l(vf, frag(&pt[0][at]), acc[r]);
    }
  float inv[RW];
  if (gate) {
#pragma unroll
    for (int r = 0; r < RW; r++) {
      float ss = acc[r][0] * acc[r][0] + acc[r][1] * acc[r][1] + acc[r][2] * acc[r][2] +
                 acc[r][3] * acc[r][3];
      ss += __shfl_xor(ss, 16);
      ss += __shfl_xor(ss, 32);
      if (hi == 0) red[ct][16 * (r0 + r) + lo] = ss;
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < RW; r++) {
      float ss = 0.f;
#pragma unroll
      for (int x = 0; x < CT; x++) ss += red[x][16 * (r0 + r) + lo];
      inv[r] = 1.f / sqrtf(ss / (float)s.V + eps);
    }
  }
  const int e = e0 + 4 * hi;
#pragma unroll
  for (int r = 0; r < RW; r++) {
    const int i = 16 * (r0 + r) + lo;
    if (i >= n || e >= s.V) continue;
    float x[4];
#pragma unroll
    for (int j = 0; j < 4; j++) x[j] = acc[r][j];
    short* dst = o + (t0 + i) * ldo + h * s.V + e;
    if (vec) {
      if (gate) {
        float g[4];
        ldv<4>(gate + (t0 + i) * ldg + h * s.V + e, g);
#pragma unroll
        for (int j = 0; j < 4; j++) x[j] *= inv[r] * silu_fast(g[j]);
      }
      stv<4>(dst, x);
    } else {
#pragma unroll
      for (int j = 0; j < 4; j++) {
        if (e + j >= s.V) continue;
        if (gate) x[j] *= inv[r] * silu_fast(ldf(gate + (t0 + i) * ldg + h * s.V + e + j));
        stf(dst + j, x[j]);
      }
    }
  }
}

// ---------------------------------------------- the same by segments
// A segment is `per` chunks of one sequence.  A workgroup walks it in steps of STEP tokens and
// keeps the state S [D, VB] in its registers, so that states pass through memory once a segment
// and not once a chunk:
//   1. linear_walk<false>: what each segment adds to the state, and its decay;
//   2. segment_scan:       the state ahead of each segment;
//   3. linear_walk<true>:  the outputs, the state going along.
// Eight waves own 16 columns of v each (64 columns: the two halves of a step's tokens besides).
// S lies as the matrix product leaves it: 4 * hi + (0 .. 3) of 16 features of one column to a
// lane, which is a fragment of two such tiles for the product with q, if q's features are read
// in that order.  The tokens of decayed k and of v, whose products need them along a lane, are
// read transposed (ds_read_tr16_b64), rows 4 * hi + (0 .. 3) and 16 on.
// Bound by instructions of all kinds, some 850 to a wave's step (SiLU, rotation, the division
// into hi and lo of q, twice k and S).  Hence no exec branches around loads and offsets of 32 bits
// from a step's first token.  The norm's exact quotient and root, as decoding has them, take 2 to 3
// % (16 sequences of 696 tokens on average, 12 heads, 136 -> 139 us): an approximate root is
// not-a-number where the squares' sum is infinite or below the smallest normal number.
// 8 sequences of 2139 tokens on average, 12 heads of 128, norm and gate in it: 170 us, by chunks 389
// (the states of 272 chunks are 214 MB); 16 of 696 140 and 233; of 32 heads, 8 of 2139, 448 and 1036.
constexpr int STEP = 32;

// Sequence b's segments have the numbers first[b] / per + b on, some of which stay unused.
DEVINL bool segment(const Chunks& ch, int B, int per, int g, int& c0, int& c1) {
  int b = 0, last = B - 1;
  while (b < last) {
    const int mid = (b + last + 1) / 2;
    if (ch.first[mid] / per + mid <= g) b = mid;
    else last = mid - 1;
  }
  c0 = ch.first[b] + (g - (ch.first[b] / per + b)) * per;
  c1 = min(c0 + per, ch.first[b + 1]);
  return c0 < c1;
}

// tokens 4 * hi + (0 .. 3) and 16 on of columns c0 + lane % 16 of a [STEP][ld] tile
DEVINL bf16x8l tokens_frag(const short* tile, int ld, int c0, int lane) {
  typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
  const short* a = tile + ((lane >> 4) * 4 + ((lane & 15) >> 2)) * ld + c0 + (lane & 3) * 4;
  union { s16x4 h[2]; bf16x8l f; } u;
  u.h[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)a);
  u.h[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(a + 16 * ld));
  return u.f;
}
// elements 4 * hi + (0 .. 3) and 16 on of a row
DEVINL bf16x8l spread_frag(const short* row, int hi) {
  union { s16x4 h[2]; bf16x8l f; } u;
  u.h[0] = *reinterpret_cast<const s16x4*>(row + 4 * hi);
  u.h[1] = *reinterpret_cast<const s16x4*>(row + 16 + 4 * hi);
  return u.f;
}

struct Hilo { unsigned hi[2], lo[2]; };        // four numbers as hi + lo
DEVINL Hilo divide(const float* x) {
  Hilo r;
#pragma unroll
  for (int j = 0; j < 2; j++) {
    r.hi[j] = pack2bf(x[2 * j], x[2 * j + 1]);
    r.lo[j] = pack2bf(x[2 * j] - __uint_as_float(r.hi[j] << 16),
                      x[2 * j + 1] - __uint_as_float(r.hi[j] & 0xffff0000u));
  }
  return r;
}
DEVINL void put(short* hi, short* lo, const float* x) {
  const Hilo r = divide(x);
  *reinterpret_cast<unsigned long long*>(hi) = (unsigned long long)r.hi[1] << 32 | r.hi[0];
  *reinterpret_cast<unsigned long long*>(lo) = (unsigned long long)r.lo[1] << 32 | r.lo[0];
}

template <int DP, int VB, bool OUT>
__global__ __launch_bounds__(512, 4) void linear_walk_kernel(
    const short* __restrict__ q, const short* __restrict__ k, const short* __restrict__ v,
    Source s, Chunks ch, int B, int per, const float* __restrict__ pw, float* __restrict__ ws,
    float* __restrict__ decays, const short* __restrict__ gate, long ldg, float eps,
    short* __restrict__ o, long ldo) {
  constexpr int QS = DP + 8, TS2 = DP + 16, VS = VB + 16, PS = STEP + 8;   // LDS rows
  constexpr int DT = DP / 16, CT = VB / 16, RW = CT / 4;
  __shared__ __attribute__((aligned(16))) short qt[2][OUT ? STEP * QS : 8];
  __shared__ __attribute__((aligned(16))) short kt[2][OUT ? STEP * QS : 8];
  __shared__ __attribute__((aligned(16))) short kd[2][STEP * TS2], vt[STEP * VS];
  __shared__ __attribute__((aligned(16))) short pt[2][OUT ? STEP * PS : 8];
  __shared__ float pws[CHUNK + 1], red[OUT ? CT : 1][STEP];
  const int h = blockIdx.y, v0 = blockIdx.z * VB;
  int c, c1;
  if (!segment(ch, B, per, blockIdx.x, c, c1)) return;
  if (threadIdx.x <= CHUNK) pws[threadIdx.x] = pw[h * (CHUNK + 1) + threadIdx.x];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int lo = lane & 15, hi = lane >> 4;
  const int ct = w % CT, r0 = (w / CT) * RW;
  const int e0 = v0 + 16 * ct;

  // the state ahead: column e0 + lo, features 16 * dt + 4 * hi + (0 .. 3)
  float* u = ws + (((long)blockIdx.x * s.H + h) * s.V + min(e0 + lo, s.V - 1)) * DP + 4 * hi;
  f32x4 S[DT];
#pragma unroll
  for (int dt = 0; dt < DT; dt++) {
    S[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (OUT && e0 + lo < s.V) S[dt] = *reinterpret_cast<const f32x4*>(u + 16 * dt);
  }

  // what this thread stages: two runs of a token's q and k, eight columns of a token's v
  const int qj = threadIdx.x / (DP / 8), qg = threadIdx.x % (DP / 8);
  const int vj = threadIdx.x / (VB / 8), ve = threadIdx.x % (VB / 8) * 8;
  const int half = s.rdims >> 1;
  const bool rot = 4 * qg < half;
  int ea, eb;
  if (s.interleaved || !rot) {
    ea = rot || s.interleaved ? 8 * qg : s.rdims + 2 * (4 * qg - half);
    eb = ea + 4;
  } else {
    ea = 4 * qg;
    eb = half + 4 * qg;
  }
  // Offsets in bytes from a step's first token, which is the same for all threads.  Threads
  // past a tile or a row's end read its first.
  const bool mine = STEP * DP / 8 == 512 || qj < STEP, myv = STEP * VB / 8 == 512 || vj < STEP;
  const bool la = mine && ea < s.D, lb = mine && eb < s.D;
  const bool va = myv && v0 + ve < s.V, vb = myv && v0 + ve + 4 < s.V;
  const bool whole = s.D == DP && v0 + VB <= s.V && STEP * DP / 8 == 512 && STEP * VB / 8 == 512;
  const unsigned ld2 = (unsigned)s.ld * 2;
  const s16x4 none{0, 0, 0, 0};
  s16x4 raw[6];
  f32x4 cs{}, sn{};
  auto fetch = [&](long t0, int n) __attribute__((always_inline)) {
    const char* kb = (const char*)(k + t0 * s.ld + h * s.D);
    const char* qb = (const char*)(q + t0 * s.ld + h * s.D);
    const char* vp = (const char*)(v + t0 * s.ld + h * s.V + v0);
    const char* cb = (const char*)(s.cs + t0 * s.rdims);
    const bool full = whole && n == STEP;
    const unsigned j = full || qj < n ? qj : 0, jv = full || vj < n ? vj : 0;
    const unsigned oa = j * ld2 + (full || la ? ea : 0) * 2, ob = j * ld2 + (full || lb ? eb : 0) * 2;
    const unsigned xa = jv * ld2 + (full || va ? ve : 0) * 2;
    const unsigned xb = jv * ld2 + (full || vb ? ve + 4 : 0) * 2;
    raw[2] = *reinterpret_cast<const s16x4*>(kb + oa);
    raw[3] = *reinterpret_cast<const s16x4*>(kb + ob);
    if constexpr (OUT) {
      raw[0] = *reinterpret_cast<const s16x4*>(qb + oa);
      raw[1] = *reinterpret_cast<const s16x4*>(qb + ob);
    }
    if (half) {
      const unsigned oc = (j * s.rdims + (rot ? 4 * qg : 0)) * 4;
      cs = *reinterpret_cast<const f32x4*>(cb + oc);
      sn = *reinterpret_cast<const f32x4*>(cb + oc + half * 4);
    }
    raw[4] = *reinterpret_cast<const s16x4*>(vp + xa);
    raw[5] = *reinterpret_cast<const s16x4*>(vp + xb);
  };
  // what was read of other tokens or columns
  auto clear = [&](int n) __attribute__((always_inline)) {
    if (whole && n == STEP) return;
    if (!(la && qj < n)) raw[0] = raw[2] = none;
    if (!(lb && qj < n)) raw[1] = raw[3] = none;
    if (!(va && vj < n)) raw[4] = none;
    if (!(vb && vj < n)) raw[5] = none;
  };
  auto runs = [&](int i, float* a, float* b) {
    float cc[4], ss[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
      a[j] = bf2f(raw[2 * i][j]);
      b[j] = bf2f(raw[2 * i + 1][j]);
      cc[j] = cs[j];
      ss[j] = sn[j];
    }
    shape_runs(a, b, s, rot, cc, ss);
  };

  const bool col_ok = e0 + 4 * hi < s.V;
  int at = 0, len = ch.len[c];
  long row = ch.row[c];
  float decay = 1.f;
  fetch(row, min(STEP, len));
  __syncthreads();                              // pws
  for (bool more = true; more;) {
    const long t0 = row + at;
    const int n = min(STEP, len - at);
    // Tokens up to where k decays: the step's end, whose state the next step's outputs need; without
    // outputs the chunk's, at whose first step S decays by all of it and at the others by pws[0], 1.
    // With half as many rounded decays the state's error is that by chunks: 16 heads of 96 that keep
    // up to 4096 tokens, 14578 tokens, 2.48e-6 against 64 bits, by steps 2.65e-6; the time is the same.
    const int until = OUT ? n : len - at, decayed = OUT || at == 0 ? until : 0;
    clear(n);
    if (mine) {
      float a[4], b[4];
      if constexpr (OUT) {
        runs(0, a, b);
        put(&qt[0][qj * QS + ea], &qt[1][qj * QS + ea], a);
        put(&qt[0][qj * QS + eb], &qt[1][qj * QS + eb], b);
      }
      runs(1, a, b);
#pragma unroll
      for (int j = 0; j < 4; j++) {
        a[j] *= s.kscale;
        b[j] *= s.kscale;
      }
      if constexpr (OUT) {
        put(&kt[0][qj * QS + ea], &kt[1][qj * QS + ea], a);
        put(&kt[0][qj * QS + eb], &kt[1][qj * QS + eb], b);
      }
      const float m = pws[max(until - 1 - qj, 0)];   // tokens past n are zero
#pragma unroll
      for (int j = 0; j < 4; j++) {
        a[j] *= m;
        b[j] *= m;
      }
      put(&kd[0][qj * TS2 + ea], &kd[1][qj * TS2 + ea], a);
      put(&kd[0][qj * TS2 + eb], &kd[1][qj * TS2 + eb], b);
    }
    if (myv) {
      if (s.silu) {
#pragma unroll
        for (int i = 4; i < 6; i++) {
          union { unsigned u[2]; s16x4 x; } y;
#pragma unroll
          for (int j = 0; j < 2; j++)
            y.u[j] = pack2bf(silu_fast(bf2f(raw[i][2 * j])), silu_fast(bf2f(raw[i][2 * j + 1])));
          raw[i] = y.x;
        }
      }
      *reinterpret_cast<s16x4*>(&vt[vj * VS + ve]) = raw[4];
      *reinterpret_cast<s16x4*>(&vt[vj * VS + ve + 4]) = raw[5];
    }
    at += STEP;
    if (at >= len) {
      at = 0;
      more = ++c < c1;
      if (more) {
        len = ch.len[c];
        row = ch.row[c];
      }
    }
    if (more) fetch(row + at, min(STEP, len - at));
    s16x4 gr[RW];
    if constexpr (OUT) {
      if (gate) {
        const char* gb = (const char*)(gate + t0 * ldg + h * s.V);
#pragma unroll
        for (int r = 0; r < RW; r++) {           // past the end: the first token's, not used
          const int i = 16 * (r0 + r) + lo;
          gr[r] = *reinterpret_cast<const s16x4*>(
              gb + ((unsigned)(i < n ? i : 0) * (unsigned)ldg + (col_ok ? e0 + 4 * hi : 0)) * 2);
        }
      }
    }
    __syncthreads();                            // staged
    f32x4 acc[RW];
    if constexpr (OUT) {
      // scores of one of four tiles, of tokens it with keys jt, to each of the first waves
      if (w < 4) {
        const int it = w >> 1, jt = w & 1;
        f32x4 sc{0.f, 0.f, 0.f, 0.f};
        if (jt <= it)
#pragma unroll
          for (int ks = 0; ks < DP / 32; ks++) {
            const int qa = (16 * it + lo) * QS + 32 * ks + 8 * hi;
            const int ka = (16 * jt + lo) * QS + 32 * ks + 8 * hi;
            const bf16x8l qh = frag(&qt[0][qa]), ql = frag(&qt[1][qa]);
            const bf16x8l kh = frag(&kt[0][ka]), kl = frag(&kt[1][ka]);
            sc = mfma16l(kl, qh, sc);
            sc = mfma16l(kh, ql, sc);
            sc = mfma16l(kh, qh, sc);
          }
        const int i = 16 * it + lo, j = 16 * jt + 4 * hi;
        float p[4];
#pragma unroll
        for (int r = 0; r < 4; r++) p[r] = i >= j + r ? sc[r] * pws[max(i - j - r, 0)] : 0.f;
        put(&pt[0][i * PS + j], &pt[1][i * PS + j], p);
      }
      // the state ahead of the step, times q
#pragma unroll
      for (int r = 0; r < RW; r++) acc[r] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int x = 0; x < DP / 32; x++) {
        const float a[4] = {S[2 * x][0], S[2 * x][1], S[2 * x][2], S[2 * x][3]};
        const float b[4] = {S[2 * x + 1][0], S[2 * x + 1][1], S[2 * x + 1][2], S[2 * x + 1][3]};
        const Hilo ha = divide(a), hb = divide(b);
        union { unsigned u[4]; bf16x8l f; } sh, sl;
#pragma unroll
        for (int j = 0; j < 2; j++) {
          sh.u[j] = ha.hi[j];
          sh.u[2 + j] = hb.hi[j];
          sl.u[j] = ha.lo[j];
          sl.u[2 + j] = hb.lo[j];
        }
#pragma unroll
        for (int r = 0; r < RW; r++) {
          const int qa = (16 * (r0 + r) + lo) * QS + 32 * x;
          const bf16x8l qh = spread_frag(&qt[0][qa], hi), ql = spread_frag(&qt[1][qa], hi);
          acc[r] = mfma16l(sl.f, qh, acc[r]);
          acc[r] = mfma16l(sh.f, ql, acc[r]);
          acc[r] = mfma16l(sh.f, qh, acc[r]);
        }
      }
#pragma unroll
      for (int r = 0; r < RW; r++) acc[r] *= pws[16 * (r0 + r) + lo + 1];
      __syncthreads();                          // scores
    }
    const bf16x8l vf = tokens_frag(vt, VS, 16 * ct, lane);
    if constexpr (OUT) {
#pragma unroll
      for (int r = 0; r < RW; r++) {
        const int pa = (16 * (r0 + r) + lo) * PS;
        acc[r] = mfma16l(vf, spread_frag(&pt[1][pa], hi), acc[r]);
        acc[r] = mfma16l(vf, spread_frag(&pt[0][pa], hi), acc[r]);
      }
    }
    if (!OUT || more) {                         // the state behind it
      const float f = pws[decayed];
#pragma unroll
      for (int dt = 0; dt < DT; dt++) {
        S[dt] *= f;
        S[dt] = mfma16l(tokens_frag(kd[1], TS2, 16 * dt, lane), vf, S[dt]);
        S[dt] = mfma16l(tokens_frag(kd[0], TS2, 16 * dt, lane), vf, S[dt]);
      }
      decay *= f;
    }
    if constexpr (OUT) {
      if (gate) {
#pragma unroll
        for (int r = 0; r < RW; r++) {
          float ss = acc[r][0] * acc[r][0] + acc[r][1] * acc[r][1] + acc[r][2] * acc[r][2] +
                     acc[r][3] * acc[r][3];
          ss += __shfl_xor(ss, 16);
          ss += __shfl_xor(ss, 32);
          if (hi == 0) red[ct][16 * (r0 + r) + lo] = ss;
        }
      }
    }
    __syncthreads();                            // read, and the sums of squares
    if constexpr (OUT) {
      char* ob = (char*)(o + t0 * ldo + h * s.V);
#pragma unroll
      for (int r = 0; r < RW; r++) {
        const int i = 16 * (r0 + r) + lo;
        float x[4] = {acc[r][0], acc[r][1], acc[r][2], acc[r][3]};
        if (gate) {
          float ss = 0.f;
#pragma unroll
          for (int y = 0; y < CT; y++) ss += red[y][i];
          const float inv = 1.f / sqrtf(ss / (float)s.V + eps);
#pragma unroll
          for (int j = 0; j < 4; j++) x[j] *= inv * silu_fast(bf2f(gr[r][j]));
        }
        if (i < n && col_ok) {
          const unsigned long long y =
              (unsigned long long)pack2bf(x[2], x[3]) << 32 | pack2bf(x[0], x[1]);
          *reinterpret_cast<unsigned long long*>(ob + ((unsigned)i * (unsigned)ldo + e0 + 4 * hi) * 2) = y;
        }
      }
    }
  }
  if constexpr (!OUT) {
    if (e0 + lo < s.V && r0 == 0)
#pragma unroll
      for (int dt = 0; dt < DT; dt++) *reinterpret_cast<f32x4*>(u + 16 * dt) = S[dt];
    if (threadIdx.x == 0 && blockIdx.z == 0) decays[(long)blockIdx.x * s.H + h] = decay;
  }
}

// in place: what a segment adds -> the state ahead of it; the slot is [D][V]
__global__ __launch_bounds__(256) void segment_scan_kernel(
    float* __restrict__ ws, const float* __restrict__ decays, float* __restrict__ state, Chunks ch,
    int per, const int* __restrict__ slots, const int* __restrict__ fresh, int H, int D, int V,
    int DP) {
  constexpr int AHEAD = 8;
  const int b = blockIdx.x, h = blockIdx.y;
  const int e = blockIdx.z * 256 + threadIdx.x;
  if (e >= V * DP) return;
  const int vi = e / DP, d = e % DP;
  const bool real = d < D;
  float* st = state + (((long)slots[b] * H + h) * D + (real ? d : 0)) * V + vi;
  float s = (fresh[b] || !real) ? 0.f : *st;
  const int g0 = ch.first[b] / per + b, n = (ch.first[b + 1] - ch.first[b] + per - 1) / per;
  const long step = (long)H * V * DP;
  float* p = ws + ((long)g0 * H + h) * V * DP + e;
  const float* f = decays + (long)g0 * H + h;
  for (int g = 0; g < n; g += AHEAD) {
    float x[AHEAD];
#pragma unroll
    for (int i = 0; i < AHEAD; i++) x[i] = g + i < n ? p[i * step] : 0.f;
#pragma unroll
    for (int i = 0; i < AHEAD; i++) {
      if (g + i >= n) break;
      p[i * step] = s;
      s = f[(g + i) * H] * s + x[i];
    }
    p += AHEAD * step;
  }
  if (real) *st = s;
}

// ------------------------------------------------------------- one token
// One workgroup per (sequence, head).  With a gate, the head's output is
// divided by its root mean square and multiplied by silu(gate) on the way out.
template <typename T, int VEC>
__global__ __launch_bounds__(256) void linear_decode_kernel(
    const T* __restrict__ q, const T* __restrict__ k, const T* __restrict__ v, Source s,
    const float* __restrict__ pw, float* __restrict__ state, const int* __restrict__ slots,
    const int* __restrict__ seq_lens, const T* __restrict__ gate, long ldg, float eps,
    T* __restrict__ o, long ldo) {
  extern __shared__ __attribute__((aligned(16))) float sh[];
  float* qs = sh;                 // [D]
  float* ks = qs + s.D;           // [D]
  float* red = qs + ((2 * s.D + 3) & ~3);   // [rows per pass][V], 16-B aligned
  __shared__ float scratch[4];
  const int b = blockIdx.x, h = blockIdx.y;
  const float* cs = s.cs + (long)b * s.rdims;
  for (int d = threadIdx.x; d < s.D; d += 256) {
    qs[d] = load_qk(q + b * s.ld + h * s.D, d, s, cs);
    ks[d] = load_qk(k + b * s.ld + h * s.D, d, s, cs) * s.kscale;
  }
  __syncthreads();
  const int nv = s.V / VEC, R = 256 / nv;
  const int r0 = threadIdx.x / nv, e0 = (threadIdx.x % nv) * VEC;
  const bool fresh = seq_lens[b] == 1;
  const float decay = pw[h * (CHUNK + 1) + 1];
  float* st = state + ((long)slots[b] * s.H + h) * s.D * s.V;
  float acc[VEC] = {};
  if (r0 < R) {
    float vv[VEC];
#pragma unroll
    for (int i = 0; i < VEC; i++) vv[i] = load_v(v + b * s.ld + h * s.V, e0 + i, s);
#pragma unroll 8
    for (int d = r0; d < s.D; d += R) {
      float x[VEC];
      float* p = st + (long)d * s.V + e0;
      if (fresh) {
#pragma unroll
        for (int i = 0; i < VEC; i++) x[i] = 0.f;
      } else {
        ldv<VEC>(p, x);
      }
      const float kd = ks[d], qd = qs[d];
#pragma unroll
      for (int i = 0; i < VEC; i++) {
        x[i] = decay * x[i] + kd * vv[i];
        acc[i] += qd * x[i];
      }
      stv<VEC>(p, x);
    }
    stv<VEC>(red + r0 * s.V + e0, acc);
  }
  __syncthreads();
  float ss = 0.f;
  for (int e = threadIdx.x; e < s.V; e += 256) {
    float x = 0.f;
    for (int r = 0; r < R; r++) x += red[r * s.V + e];
    red[e] = x;                    // column e is this thread's alone
    ss += x * x;
  }
  float inv = 1.f;
  if (gate) inv = 1.f / sqrtf(block_sum<256>(ss, scratch) / (float)s.V + eps);
  for (int e = threadIdx.x; e < s.V; e += 256) {
    float x = red[e] * inv;
    if (gate) x *= act_silu(ldf(gate + b * ldg + h * s.V + e));
    stf(o + b * ldo + h * s.V + e, x);
  }
}

// ======================================================== host wrappers ==
static Source make_source(const torch::Tensor& q, const torch::Tensor& k, const torch::Tensor& v,
                          const torch::Tensor& pw, const c10::optional<torch::Tensor>& cs,
                          bool interleaved, bool silu, double kscale) {
  const long H = pw.size(0);
  on_gpu({q, k, v, pw, cs});
  TORCH_CHECK(q.dim() == 2 && k.sizes() == q.sizes() && v.size(0) == q.size(0));
  TORCH_CHECK(q.stride(1) == 1 && k.stride(1) == 1 && v.stride(1) == 1 &&
              q.stride(0) == k.stride(0) && q.stride(0) == v.stride(0),
              "q, k and v are columns of one row-major projection");
  TORCH_CHECK(q.scalar_type() == k.scalar_type() && q.scalar_type() == v.scalar_type());
  TORCH_CHECK(q.size(1) % H == 0 && v.size(1) % H == 0);
  TORCH_CHECK(pw.dim() == 2 && pw.size(1) == CHUNK + 1 && pw.is_contiguous() &&
              pw.scalar_type() == torch::kFloat32, "decay powers are [heads, ", CHUNK + 1, "]");
  Source s;
  s.ld = q.stride(0);
  s.H = H;
  s.D = q.size(1) / H;
  s.V = v.size(1) / H;
  s.cs = cs.has_value() ? cs->data_ptr<float>() : nullptr;
  s.rdims = cs.has_value() ? cs->size(1) : 0;
  s.interleaved = interleaved;
  s.silu = silu;
  s.kscale = kscale;
  TORCH_CHECK(s.D >= 1 && s.D <= 256 && s.V >= 1 && s.rdims <= s.D && s.rdims % 2 == 0);
  if (cs.has_value())
    TORCH_CHECK(cs->scalar_type() == torch::kFloat32 && cs->is_contiguous() && cs->size(0) == q.size(0));
  return s;
}

static void check_state(const torch::Tensor& state, const Source& s) {
  TORCH_CHECK(state.scalar_type() == torch::kFloat32 && state.is_contiguous() && state.dim() == 4 &&
              state.size(1) == s.H && state.size(2) == s.D && state.size(3) == s.V);
}

static void check_ints(const torch::Tensor& t, long n) {
  TORCH_CHECK(t.is_cuda() && t.scalar_type() == torch::kInt && t.is_contiguous() && t.numel() == n);
}

// How many of n chunks of B sequences make a segment; 0: chunk by chunk.  Both counts are known
// here, but not how long each sequence is, so that the lines lie where neither even sequences nor
// one long one among short ones is slower than by chunks.  A workgroup's steps follow each other:
// segments stay near the time that all of them take (`work` chunks on 512 workgroups, two to a CU),
// for one long sequence takes its segment's steps however many CUs are idle (200 of 20 tokens and
// one of 2560, 12 heads: 645 us with 3 chunks, 621 with 4, 790 with 24, by chunks 725).  Up to that
// as many as leave one round, if three quarters of a segment are lost at each sequence's end (half
// of one is, most times): 16 sequences of 696 on average, 12 heads, 147 us with 3, 140 with 6; 8 of
// 2139 198 with 3, 170 with 8.  Where these are more rounds, 6, or of long sequences the number
// with which the rounds are through soonest: 32 heads, 190 chunks of one 281 with 6, 268 with 12.
//
// By chunks / so, us, heads of 128: with a CU to each workgroup, 12 heads, one of 1004 tokens
// 37 / 32; without, but no more than two, which leaves no round to save, one of 2028 (384) 48 / 46,
// 32 heads, one of 1004 (512) 51 / 55; 12 heads, one of 2693 (516) 71 / 58, of 6124 113 / 82.  Of
// fewer than 2.5 chunks to a sequence there is little to save, and only many of them save it: 32
// heads, 48 of 108 tokens 604 / 378, 33 of 100 (32 of 40) 291 / 261, but 12 heads 109 / 118.  Heads
// of 64, whose states are a quarter: 16 heads, one of 1004 22 / 27, of 3052 42 / 38.  Of 32, 16 heads,
// 16 of 172 tokens 28 / 36, 32 of 40 and one of 4096 57 / 58 to 62: by chunks.
long linear_attn_segment(long n, long B, long H, long D, long V) {
  if (D <= 32 || D > 128) return 0;
  const long columns = V <= 64 ? 64 : 128, across = H * ((V + columns - 1) / columns);
  const long work = n * across;
  if (2 * n < 5 * B) return D > 64 && 4 * n >= 5 * B && work >= 2048 ? 4 : 0;
  if (D <= 64 ? work < 640 : work <= 512 && (work < 144 || work + B * across > 256)) return 0;
  auto groups = [&](long i) { return across * (4 * n + 3 * B * (i - 1)) / (4 * i); };
  const long most = std::min(12L, (5 * work + 2047) / 2048);
  long per = 1;
  while (per < most && groups(per) > 512) per++;
  if (groups(per) > 512) {
    per = std::min(per, 6L);
    auto cost = [&](long i) { return (groups(i) + 511) / 512 * (2 * i + 1); };
    if (n >= 24 * B)
      for (long i = 6; i <= 24; i++)
        if (cost(i) < cost(per)) per = i;
  }
  return per;
}

// o [T, H * V] (any row stride) <- portions described by chunks (int32 [3, n]:
// sequence, first row, length), first (int32 [B + 1]), slots and fresh (int32
// [B]).  With a gate, each head's output is divided by its root mean square and
// multiplied by silu(gate): bf16 and V <= 128 only.
void linear_attn_chunked(torch::Tensor q, torch::Tensor k, torch::Tensor v, torch::Tensor pw,
                         c10::optional<torch::Tensor> cs, bool interleaved, bool silu,
                         double kscale, torch::Tensor chunks, torch::Tensor first,
                         torch::Tensor slots, torch::Tensor fresh, torch::Tensor state,
                         c10::optional<torch::Tensor> gate, double eps, torch::Tensor o) {
  const Source s = make_source(q, k, v, pw, cs, interleaved, silu, kscale);
  check_state(state, s);
  on_gpu({state, gate, o});
  const long n = chunks.size(1), B = slots.numel();
  check_ints(chunks, 3 * n);
  check_ints(first, B + 1);
  check_ints(slots, B);
  check_ints(fresh, B);
  TORCH_CHECK(o.stride(1) == 1 && o.scalar_type() == q.scalar_type() && o.size(0) == q.size(0) &&
              o.size(1) == (long)s.H * s.V);
  if (gate.has_value())
    TORCH_CHECK(q.scalar_type() == torch::kBFloat16 && s.V <= 128 && gate->stride(1) == 1 &&
                gate->scalar_type() == q.scalar_type() && gate->sizes() == o.sizes());
  if (n == 0) return;
  const int DP = s.D <= 32 ? 32 : s.D <= 64 ? 64 : s.D <= 128 ? 128 : 256;
  const bool split = q.scalar_type() == torch::kBFloat16;
  int* cp = chunks.data_ptr<int>();
  const Chunks ch{cp, cp + n, cp + 2 * n, first.data_ptr<int>()};
  auto stream = at::hip::getCurrentHIPStream();
  const dim3 grid(n, s.H, (s.V + VBLK - 1) / VBLK);
  const int DV = s.D * s.V;
  const float* pwp = pw.data_ptr<float>();
  torch::Tensor ws;
  if (split) {
    auto al = [](const void* p) { return ((uintptr_t)p % 8) == 0; };
    const bool vec = s.D % 4 == 0 && s.V % 4 == 0 && s.rdims % 8 == 0 && s.ld % 4 == 0 &&
                     o.stride(0) % 4 == 0 && al(q.data_ptr()) && al(k.data_ptr()) &&
                     al(v.data_ptr()) && al(o.data_ptr()) && ((uintptr_t)s.cs % 16) == 0 &&
                     (!gate.has_value() || (gate->stride(0) % 4 == 0 && al(gate->data_ptr())));
    const short* gp = gate.has_value() ? (const short*)gate->data_ptr() : nullptr;
    const long ldg = gate.has_value() ? gate->stride(0) : 0;
    auto short_rows = [](long ld) { return ld >= 0 && ld < 1L << 24; };   // a step's offsets: 32 bits
    const int per = linear_attn_segment(n, B, s.H, s.D, s.V);
    if (vec && per && short_rows(s.ld) && short_rows(ldg) && short_rows(o.stride(0)) &&
        s.rdims < 1 << 24) {
      const long G = n / per + B;
      auto parts = torch::empty({G, s.H, s.V, DP}, state.options());
      auto decays = torch::empty({G, s.H}, state.options());
      float* wp = parts.data_ptr<float>();
      float* dp = decays.data_ptr<float>();
#define WALK(DD, VB)                                                                            \
  do {                                                                                          \
    const dim3 sg(G, s.H, (s.V + VB - 1) / VB);                                                 \
    hipLaunchKernelGGL((linear_walk_kernel<DD, VB, false>), sg, dim3(512), 0, stream,           \
                       (const short*)q.data_ptr(), (const short*)k.data_ptr(),                  \
                       (const short*)v.data_ptr(), s, ch, (int)B, per, pwp, wp, dp, nullptr,    \
                       0L, 0.f, nullptr, 0L);                                                   \
    hipLaunchKernelGGL(segment_scan_kernel, dim3(B, s.H, (s.V * DD + 255) / 256), dim3(256), 0, \
                       stream, wp, dp, state.data_ptr<float>(), ch, per, slots.data_ptr<int>(), \
                       fresh.data_ptr<int>(), s.H, s.D, s.V, DD);                               \
    hipLaunchKernelGGL((linear_walk_kernel<DD, VB, true>), sg, dim3(512), 0, stream,            \
                       (const short*)q.data_ptr(), (const short*)k.data_ptr(),                  \
                       (const short*)v.data_ptr(), s, ch, (int)B, per, pwp, wp, dp, gp, ldg,    \
                       (float)eps, (short*)o.data_ptr(), (long)o.stride(0));                    \
  } while (0)
#define WALK_V(DD) do { if (s.V <= 64) WALK(DD, 64); else WALK(DD, 128); } while (0)
      if (DP == 64) WALK_V(64);
      else WALK_V(128);
#undef WALK_V
#undef WALK
      HIP_CHECK_LAST();
      return;
    }
    ws = torch::empty({n, s.H, s.V, DP}, state.options());
    float* wsp = ws.data_ptr<float>();
#define SPLIT(DD, VB)                                                                           \
  do {                                                                                          \
    const dim3 sg(n, s.H, (s.V + VB - 1) / VB);                                                 \
    hipLaunchKernelGGL((chunk_state_split_kernel<DD, VB>), sg, dim3(512), 0, stream,            \
                       (const short*)k.data_ptr(), (const short*)v.data_ptr(), s, ch, pwp, wsp, \
                       vec);                                                                    \
    hipLaunchKernelGGL(chunk_scan_split_kernel, dim3(B, s.H, (s.V * DD + 255) / 256),           \
                       dim3(256), 0, stream, wsp, state.data_ptr<float>(), ch,                  \
                       slots.data_ptr<int>(), fresh.data_ptr<int>(), pwp, s.H, s.D, s.V, DD);   \
    hipLaunchKernelGGL((chunk_out_split_kernel<DD, VB>), sg, dim3(512), 0, stream,              \
                       (const short*)q.data_ptr(), (const short*)k.data_ptr(),                  \
                       (const short*)v.data_ptr(), s, ch, pwp, (const unsigned*)wsp, gp, ldg,   \
                       (float)eps, (short*)o.data_ptr(), (long)o.stride(0), vec);               \
  } while (0)
#define SPLIT_V(DD) do { if (s.V <= 64) SPLIT(DD, 64); else SPLIT(DD, 128); } while (0)
    if (DP == 32) SPLIT_V(32);
    else if (DP == 64) SPLIT_V(64);
    else if (DP == 128) SPLIT_V(128);
    else SPLIT_V(256);
#undef SPLIT_V
#undef SPLIT
    HIP_CHECK_LAST();
    return;
  }
  TORCH_CHECK(q.scalar_type() == torch::kFloat32);
  ws = torch::empty({n, s.H, s.V, s.D}, state.options());
  float* wsp = ws.data_ptr<float>();
#define PHASES(DD)                                                                             \
  do {                                                                                         \
    hipLaunchKernelGGL((chunk_state_kernel<float, DD>), grid, dim3(256), 0, stream,            \
                       (const float*)k.data_ptr(), (const float*)v.data_ptr(), s, ch, pwp, wsp); \
    hipLaunchKernelGGL(chunk_scan_kernel, dim3(B, s.H, (DV + 255) / 256), dim3(256), 0, stream, \
                       wsp, state.data_ptr<float>(), ch, slots.data_ptr<int>(),                \
                       fresh.data_ptr<int>(), pwp, s.H, DV);                                   \
    hipLaunchKernelGGL((chunk_out_kernel<float, DD>), grid, dim3(256), 0, stream,              \
                       (const float*)q.data_ptr(), (const float*)k.data_ptr(),                 \
                       (const float*)v.data_ptr(), s, ch, pwp, wsp, (float*)o.data_ptr(),      \
                       (long)o.stride(0));                                                     \
  } while (0)
  if (DP == 32) PHASES(32);
  else if (DP == 64) PHASES(64);
  else if (DP == 128) PHASES(128);
  else PHASES(256);
#undef PHASES
  HIP_CHECK_LAST();
}

// o [B, H * V] (any row stride) <- one token of each of B sequences
void linear_attn_decode(torch::Tensor q, torch::Tensor k, torch::Tensor v, torch::Tensor pw,
                        c10::optional<torch::Tensor> cs, bool interleaved, bool silu,
                        double kscale, torch::Tensor slots, torch::Tensor seq_lens,
                        torch::Tensor state, c10::optional<torch::Tensor> gate, double eps,
                        torch::Tensor o) {
  const Source s = make_source(q, k, v, pw, cs, interleaved, silu, kscale);
  check_state(state, s);
  on_gpu({state, gate, o});
  const long B = q.size(0);
  check_ints(slots, B);
  check_ints(seq_lens, B);
  TORCH_CHECK(o.scalar_type() == q.scalar_type() && o.size(0) == B && o.stride(1) == 1 &&
              o.size(1) == (long)s.H * s.V);
  if (gate.has_value())
    TORCH_CHECK(gate->scalar_type() == q.scalar_type() && gate->size(0) == B &&
                gate->stride(1) == 1 && gate->size(1) == o.size(1));
  if (B == 0) return;
  const bool vec = s.V % 4 == 0;
  TORCH_CHECK(s.V / (vec ? 4 : 1) <= 256, "value width too large");
  const int R = 256 / (s.V / (vec ? 4 : 1));
  const size_t lds = sizeof(float) * (((2 * s.D + 3) & ~3) + (long)R * s.V);
  auto stream = at::hip::getCurrentHIPStream();
#define LAUNCH(TT, VEC)                                                                         \
  hipLaunchKernelGGL((linear_decode_kernel<TT, VEC>), dim3(B, s.H), dim3(256), lds, stream,     \
                     (const TT*)q.data_ptr(), (const TT*)k.data_ptr(), (const TT*)v.data_ptr(), \
                     s, pw.data_ptr<float>(), state.data_ptr<float>(), slots.data_ptr<int>(),   \
                     seq_lens.data_ptr<int>(),                                                  \
                     gate.has_value() ? (const TT*)gate->data_ptr() : nullptr,                  \
                     gate.has_value() ? (long)gate->stride(0) : 0L, (float)eps,                 \
                     (TT*)o.data_ptr(), (long)o.stride(0))
  if (q.scalar_type() == torch::kBFloat16) {
    if (vec) LAUNCH(short, 4); else LAUNCH(short, 1);
  } else {
    TORCH_CHECK(q.scalar_type() == torch::kFloat32);
    if (vec) LAUNCH(float, 4); else LAUNCH(float, 1);
  }
#undef LAUNCH
  HIP_CHECK_LAST();
}
