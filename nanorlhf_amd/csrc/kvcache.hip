// Paged KV-cache ops: append + single-token decode attention (MFMA).
//
// Layouts: K cache [P, ps, Hkv, D] (token-major rows); V cache d-major per
// page, [P, Hkv, D, ps], so the decode PV MFMA B-fragment (contraction over
// tokens) is a contiguous 16-B load.  page_size MUST be 16 (one MFMA
// half-K per page half).
//
// paged_attn_decode: one 256-thread workgroup (4 waves) per (sequence, kv-head,
// split of the context).  The G <= 16 grouped query heads are the 16 columns of
// v_mfma_f32_16x16x32 tiles (S^T = K Q^T, O^T += V^T P^T), so a lane's scores
// are all of one head and the online softmax needs two exchanges between lanes;
// each wave walks 32-token KV tiles with stride 4.  Waves merge through LDS,
// splits through a second small kernel.
#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>

#include "common.h"
#include "checks.h"
#include "qkv.h"

typedef __bf16 bf16x8k __attribute__((ext_vector_type(8)));
typedef int i32x2k __attribute__((ext_vector_type(2)));
typedef int i32x4k __attribute__((ext_vector_type(4)));

DEVINL f32x4 mfma16k(bf16x8k a, bf16x8k b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

DEVINL f32x4 mfma16k_fp8(long a, long b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_fp8_fp8(a, b, c, 0, 0, 0);
}

// ---- OCP fp8 e4m3 KV support (gfx950-native cvt instructions) ----------
DEVINL unsigned char f32_to_fp8(float x) {
  return (unsigned char)(__builtin_amdgcn_cvt_pk_fp8_f32(x, x, 0, false) & 0xff);
}

// quantize 8 f32 to 8 packed fp8 bytes (for Q / P operands on the fp8 path)
DEVINL long pack8_fp8(const float* f) {
  int w0 = __builtin_amdgcn_cvt_pk_fp8_f32(f[0], f[1], 0, false);
  w0 = __builtin_amdgcn_cvt_pk_fp8_f32(f[2], f[3], w0, true);
  int w1 = __builtin_amdgcn_cvt_pk_fp8_f32(f[4], f[5], 0, false);
  w1 = __builtin_amdgcn_cvt_pk_fp8_f32(f[6], f[7], w1, true);
  i32x2k w;
  w[0] = w0;
  w[1] = w1;
  return *reinterpret_cast<long*>(&w);
}

// ------------------------------------------------------------- kv append
template <typename CT>
__global__ void kv_append_kernel(const short* __restrict__ k,
                                 const short* __restrict__ v,
                                 const long* __restrict__ slots,
                                 CT* __restrict__ kc,
                                 CT* __restrict__ vc,
                                 long T, int Hkv, int D, int ps) {
  const int row_elems = Hkv * D;
  long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;  // units of 8 elems
  const int nvec = row_elems / 8;
  if (idx >= T * (long)nvec) return;
  const long t = idx / nvec;
  const int e0 = (int)(idx % nvec) * 8;
  const long slot = slots[t];
  s16x8 kk = *reinterpret_cast<const s16x8*>(k + t * (long)row_elems + e0);
  s16x8 vv = *reinterpret_cast<const s16x8*>(v + t * (long)row_elems + e0);
  const long page = slot / ps;
  const int off = (int)(slot % ps);
  const int h = e0 / D;
  const int d0 = e0 % D;
  if constexpr (sizeof(CT) == 2) {
    // K: token-major row copy (bf16)
    *reinterpret_cast<s16x8*>(kc + slot * (long)row_elems + e0) = kk;
#pragma unroll
    for (int j = 0; j < 8; j++)
      vc[((page * Hkv + h) * (long)D + d0 + j) * ps + off] = (CT)vv[j];
  } else {
    // fp8 e4m3 quantized cache.  K is stored FRAGMENT-MAJOR within each
    // token's D block: byte group (c = d0/32, hi = (d0%32)/8) lands at
    // hi*(D/4) + c*8, so the decode QK^T reads its per-c 8-byte MFMA
    // fragments as one contiguous 16-B load per c-PAIR (the natural
    // [d] order would leave half-width 8-B loads on the K stream).
    const int c = d0 >> 5, hi8 = (d0 >> 3) & 3;
    const int kd0 = hi8 * (D >> 2) + c * 8;
#pragma unroll
    for (int j = 0; j < 8; j++) {
      kc[slot * (long)row_elems + h * D + kd0 + j] = (CT)f32_to_fp8(bf2f(kk[j]));
      vc[((page * Hkv + h) * (long)D + d0 + j) * ps + off] =
          (CT)f32_to_fp8(bf2f(vv[j]));
    }
  }
}

void kv_append(torch::Tensor k, torch::Tensor v, torch::Tensor slots,
               torch::Tensor k_cache, torch::Tensor v_cache) {
  on_gpu({k, v, slots, k_cache, v_cache});
  TORCH_CHECK(k.scalar_type() == torch::kBFloat16 && k.is_contiguous());
  TORCH_CHECK(slots.scalar_type() == torch::kLong);
  const long T = k.size(0);
  if (T == 0) return;
  const int Hkv = k.size(1), D = k.size(2);
  const int ps = k_cache.size(1);
  TORCH_CHECK(D % 8 == 0);
  const long total = T * (Hkv * D / 8);
  auto stream = at::hip::getCurrentHIPStream();
  if (k_cache.scalar_type() == torch::kBFloat16) {
    hipLaunchKernelGGL(kv_append_kernel<short>, dim3((total + 255) / 256), dim3(256),
                       0, stream,
                       (const short*)k.data_ptr(), (const short*)v.data_ptr(),
                       slots.data_ptr<long>(), (short*)k_cache.data_ptr(),
                       (short*)v_cache.data_ptr(), T, Hkv, D, ps);
  } else if (k_cache.scalar_type() == torch::kFloat8_e4m3fn) {
    hipLaunchKernelGGL(kv_append_kernel<unsigned char>, dim3((total + 255) / 256),
                       dim3(256), 0, stream,
                       (const short*)k.data_ptr(), (const short*)v.data_ptr(),
                       slots.data_ptr<long>(), (unsigned char*)k_cache.data_ptr(),
                       (unsigned char*)v_cache.data_ptr(), T, Hkv, D, ps);
  } else {
    TORCH_CHECK(false, "kv cache must be bf16 or fp8_e4m3fn");
  }
  HIP_CHECK_LAST();
}

static void check_qkv(const torch::Tensor& qkv, const torch::Tensor& table,
                      const torch::Tensor& positions, const torch::Tensor& slots,
                      const torch::Tensor& k_cache, const torch::Tensor& v_cache, long Hq,
                      const c10::optional<torch::Tensor>& bias) {
  on_gpu({qkv, table, positions, slots, k_cache, v_cache, bias});
  const bool parts = qkv.dim() == 3;
  TORCH_CHECK(qkv.is_contiguous() &&
              (parts ? qkv.scalar_type() == torch::kFloat32 && qkv.size(0) > 0 && qkv.size(0) <= 8
                     : qkv.scalar_type() == torch::kBFloat16 && qkv.dim() == 2 && !bias));
  TORCH_CHECK(k_cache.dim() == 4 && k_cache.is_contiguous() && v_cache.is_contiguous() &&
              v_cache.scalar_type() == k_cache.scalar_type());
  const long T = qkv.size(-2), N = qkv.size(-1), ps = k_cache.size(1), Hkv = k_cache.size(2),
             D = k_cache.size(3);
  TORCH_CHECK(Hq > 0 && N == (Hq + 2 * Hkv) * D && D % 32 == 0);
  if (bias)
    TORCH_CHECK(bias->scalar_type() == torch::kBFloat16 && bias->is_contiguous() &&
                bias->numel() == N, "bias must be bf16, one per column");
  TORCH_CHECK(v_cache.size(1) == Hkv && v_cache.size(2) == D && v_cache.size(3) == ps);
  TORCH_CHECK(table.scalar_type() == torch::kFloat32 && table.is_contiguous() &&
              table.size(-1) == D, "rope table must be fp32 [positions, head_dim]");
  TORCH_CHECK(positions.scalar_type() == torch::kLong && positions.is_contiguous() &&
              positions.numel() == T, "positions must be int64, one per token");
  TORCH_CHECK(slots.scalar_type() == torch::kLong && slots.is_contiguous() && slots.numel() == T);
  TORCH_CHECK(k_cache.scalar_type() == torch::kFloat8_e4m3fn ||
              k_cache.scalar_type() == torch::kBFloat16, "kv cache must be bf16 or fp8_e4m3fn");
}

// qkv [T, (Hq + 2 Hkv) D]: q and k rotated, k and v into the cache at `slots`.
// Returns q [T, Hq, D], and k and v [T, Hkv, D] if asked for.  Or qkv float32 [splits, T, ..],
// parts of a projection that this adds up, with its bias.
std::vector<torch::Tensor> qkv_rope_append(torch::Tensor qkv, torch::Tensor table,
                                           torch::Tensor positions, torch::Tensor slots,
                                           torch::Tensor k_cache, torch::Tensor v_cache, long Hq,
                                           bool want_kv, c10::optional<torch::Tensor> bias) {
  check_qkv(qkv, table, positions, slots, k_cache, v_cache, Hq, bias);
  const bool parts = qkv.dim() == 3;
  const long T = qkv.size(-2), N = qkv.size(-1), ps = k_cache.size(1), Hkv = k_cache.size(2),
             D = k_cache.size(3);
  if ((uintptr_t)qkv.data_ptr() % 16) qkv = qkv.clone();
  if (bias && (uintptr_t)bias->data_ptr() % 16) bias = bias->clone();
  const auto opt = qkv.options().dtype(torch::kBFloat16);
  auto q = torch::empty({T, Hq, D}, opt);
  std::vector<torch::Tensor> out{q};
  if (want_kv)
    for (int i = 0; i < 2; i++) out.push_back(torch::empty({T, Hkv, D}, opt));
  auto stream = at::hip::getCurrentHIPStream();
  const bool fp8 = k_cache.scalar_type() == torch::kFloat8_e4m3fn;
  by_tokens(T, (Hq + 2 * Hkv) * (D / 16), [&](long t0, unsigned units) {
    QkvRope a{};
    if (parts) {
      a.parts = qkv.data_ptr<float>() + t0 * N;
      a.part = T * N;
      a.splits = qkv.size(0);
      a.bias = bias ? (const short*)bias->data_ptr() : nullptr;
    } else {
      a.qkv = (const short*)qkv.data_ptr() + t0 * N;
    }
    a.q = (short*)q.data_ptr() + t0 * Hq * D;
    if (want_kv) {
      a.k = (short*)out[1].data_ptr() + t0 * Hkv * D;
      a.v = (short*)out[2].data_ptr() + t0 * Hkv * D;
    }
    a.table = table.data_ptr<float>();
    a.pos = positions.data_ptr<long>() + t0;
    a.slots = slots.data_ptr<long>() + t0;
    a.kc = k_cache.data_ptr();
    a.vc = v_cache.data_ptr();
    a.Hq = Hq;
    a.Hkv = Hkv;
    a.D = D;
    a.ps = ps;
    const dim3 block(qkv_block(units)), grid((units + block.x - 1) / block.x);
#define LAUNCH(CT, P) hipLaunchKernelGGL((qkv_rope_kernel<CT, P>), grid, block, 0, stream, a, units)
    if (fp8) { if (parts) LAUNCH(unsigned char, true); else LAUNCH(unsigned char, false); }
    else { if (parts) LAUNCH(short, true); else LAUNCH(short, false); }
#undef LAUNCH
  });
  HIP_CHECK_LAST();
  return out;
}

// ------------------------------------------------------- decode attention
// Mask and output options of the general form (EXT); the plain form compiles
// them away.
struct DecodeExt {
  int size;          // sliding window: position i sees j with i - j < size ...
  int keep;          // ... and every j < keep
  int V;             // value width of the output (<= DV, the cache's)
  long ldo;          // output row stride
  const float* uncs; // [B, V] cos | sin: turn the output's pairs (2m, 2m+1) back
  int gchunks;       // query-head groups of 16 per kv head
};

// What bounds it: reading the cache.  K of the next tile and V of this one are
// in flight while a tile's scores are worked on; a wave that asked for its page,
// its K and its V one after the other had 5 us per tile of 32 tokens to wait.
// 16 tokens of two pages, as MFMA fragments
template <int D, typename CT>
struct KTile {
  static constexpr int BYTES = D * (int)sizeof(CT) / 4;          // per lane and 16 tokens
  static constexpr int NV = BYTES >= 16 ? BYTES / 16 : 1;
  i32x4k r[2][NV];
  // lane (hi, lo): token lo of page n; bf16: elements 32c + 8hi .. + 7 of every
  // c, fp8: the fragment-major D / 4 bytes of hi
  DEVINL void load(const CT* kc, int page0, int page1, int Hkv, int kvh, int lo, int hi) {
#pragma unroll
    for (int n = 0; n < 2; n++) {
      const CT* row = kc + (((long)(n ? page1 : page0) * 16 + lo) * Hkv + kvh) * D;
      if constexpr (sizeof(CT) == 2) {
#pragma unroll
        for (int c = 0; c < NV; c++)
          r[n][c] = *reinterpret_cast<const i32x4k*>(row + 32 * c + 8 * hi);
      } else if constexpr (BYTES >= 16) {
#pragma unroll
        for (int c = 0; c < NV; c++)
          r[n][c] = *reinterpret_cast<const i32x4k*>(row + hi * (D / 4) + 16 * c);
      } else {
        const i32x2k w = *reinterpret_cast<const i32x2k*>(row + hi * (D / 4));
        r[n][0] = i32x4k{w[0], w[1], 0, 0};
      }
    }
  }
};

// a, b hold, in the lanes of group hi (of four), something of tokens 4 * hi ..
// + 3 of the first and of the second page; afterwards of tokens 8 * hi .. + 3 and
// 8 * hi + 4 .. + 7 of the 32
DEVINL void tokens_to_k(unsigned& a, unsigned& b) {
  auto x = __builtin_amdgcn_permlane32_swap(a, b, false, false);
  auto y = __builtin_amdgcn_permlane16_swap(x[0], x[1], false, false);
  a = y[0];
  b = y[1];
}

// over the four groups of 16 lanes
DEVINL float max_groups(float x) {
  x = fmaxf(x, __shfl_xor(x, 16));
  return fmaxf(x, __shfl_xor(x, 32));
}
DEVINL float sum_groups(float x) {
  x += __shfl_xor(x, 16);
  return x + __shfl_xor(x, 32);
}

// tiles of 32 tokens with a visible key: those of the kept first tokens, then
// the window's
struct TileRange { int win_lo, win_tile, kept, n; };
template <bool EXT>
DEVINL TileRange tile_range(int L, const DecodeExt& ext) {
  TileRange t;
  t.win_lo = EXT ? max(0, L - ext.size) : 0;
  t.win_tile = t.win_lo / 32;
  t.kept = EXT ? min((ext.keep + 31) / 32, t.win_tile) : 0;
  t.n = t.kept + (L + 31) / 32 - t.win_tile;
  return t;
}

// o[0], o[1] at columns d, d + 1 of head h of row b, times inv, turned back if asked
template <bool EXT>
DEVINL void write_pair(short* out, float o0, float o1, int b, int h, int d, int Hq, int DV,
                       const DecodeExt& ext) {
  if constexpr (EXT) {
    if (ext.uncs && d < ext.V) {
      const float* cs = ext.uncs + (long)b * ext.V;
      const float c = cs[d >> 1], s = cs[ext.V / 2 + (d >> 1)];
      const float t = o0 * c + o1 * s;
      o1 = o1 * c - o0 * s;
      o0 = t;
    }
    short* op = out + (long)b * ext.ldo + (long)h * ext.V + d;
    if (d < ext.V) op[0] = f2bf(o0);
    if (d + 1 < ext.V) op[1] = f2bf(o1);
  } else {
    const unsigned w = (unsigned)(unsigned short)f2bf(o0) | (unsigned)(unsigned short)f2bf(o1) << 16;
    *reinterpret_cast<unsigned*>(out + ((long)b * Hq + h) * DV + d) = w;
  }
}

// What a decode step's projection leaves to be done before its attention: the sequence's new
// q, k and v are added up, rotated and cached as qkv_rope_kernel does it.
// A workgroup makes those of its kv head and its query heads, which it keeps in LDS: keys and
// values of the newest token are put into its tile from there, so that no workgroup reads what
// another one may still be writing.  One launch and one wait for the projection where there
// were two, in us: 64 x 170 tokens of 12 over 2 heads in fp8 9.0 -> 6.8, one sequence of 60
// tokens 7.4 -> 5.7, 32 x 2000 in bf16 17.9 -> 15.4, 256 x 600 24.8 -> 22.4.
template <int D, typename CT>
struct alignas(16) NewToken {         // read and written 16 bytes at a time
  short q[16][D], k[D], v[D];
  unsigned char k8[D], v8[D];       // of an fp8 cache; k8 fragment-major, as the cache has it

  // thread `unit` of (G + 2) * D / 16
  DEVINL void make(const QkvRope& a, int b, int kvh, int G, int unit, bool store) {
    const int g = unit % (D / 16), i = unit / (D / 16);      // i < G: query, G: key, G + 1: value
    const int h = i < G ? kvh * G + i : i == G ? a.Hq + kvh : a.Hq + a.Hkv + kvh;
    const int d1 = 8 * g, d2 = D / 2 + 8 * g;
    const long row = (long)b * (a.Hq + 2 * a.Hkv) + h, pos = a.pos[b], slot = a.slots[b];
    s16x8 x1, x2;
    if (a.parts) {
      const float* src = a.parts + row * D;
      const short* bias = a.bias ? a.bias + h * D : nullptr;
      x1 = sum_parts8(src + d1, a.part, a.splits, bias ? bias + d1 : nullptr);
      x2 = sum_parts8(src + d2, a.part, a.splits, bias ? bias + d2 : nullptr);
    } else {
      x1 = *reinterpret_cast<const s16x8*>(a.qkv + row * D + d1);
      x2 = *reinterpret_cast<const s16x8*>(a.qkv + row * D + d2);
    }
    if (i <= G) rotate8(x1, x2, a.table + pos * D + d1, D, 1.f, x1, x2);
    short* to = i < G ? q[i] : i == G ? k : v;
    *reinterpret_cast<s16x8*>(to + d1) = x1;
    *reinterpret_cast<s16x8*>(to + d2) = x2;
    if (i < G) return;
    const uint2 w1 = make_uint2(fp8x4(x1, 0), fp8x4(x1, 4));
    const uint2 w2 = make_uint2(fp8x4(x2, 0), fp8x4(x2, 4));
    if (i == G) {
      CT* kc = (CT*)a.kc + (slot * a.Hkv + kvh) * D;
      if constexpr (sizeof(CT) == 2) {
        if (store) {
          *reinterpret_cast<s16x8*>(kc + d1) = x1;
          *reinterpret_cast<s16x8*>(kc + d2) = x2;
        }
      } else {
        const int at1 = ((d1 >> 3) & 3) * (D >> 2) + (d1 >> 5) * 8;
        const int at2 = ((d2 >> 3) & 3) * (D >> 2) + (d2 >> 5) * 8;
        *reinterpret_cast<uint2*>(k8 + at1) = w1;
        *reinterpret_cast<uint2*>(k8 + at2) = w2;
        if (store) {
          *reinterpret_cast<uint2*>(kc + at1) = w1;
          *reinterpret_cast<uint2*>(kc + at2) = w2;
        }
      }
    } else {
      if constexpr (sizeof(CT) == 1) {
        *reinterpret_cast<uint2*>(v8 + d1) = w1;
        *reinterpret_cast<uint2*>(v8 + d2) = w2;
      }
      if (!store) return;
      CT* vc = (CT*)a.vc + ((slot / 16 * a.Hkv + kvh) * D) * 16 + slot % 16;
#pragma unroll
      for (int j = 0; j < 8; j++) {
        if constexpr (sizeof(CT) == 2) {
          vc[(d1 + j) * 16] = x1[j];
          vc[(d2 + j) * 16] = x2[j];
        } else {
          vc[(d1 + j) * 16] = (CT)((j < 4 ? w1.x : w1.y) >> (8 * (j & 3)));
          vc[(d2 + j) * 16] = (CT)((j < 4 ? w2.x : w2.y) >> (8 * (j & 3)));
        }
      }
    }
  }
};
struct NoToken {};

// blockIdx.x = (sequence, kv head, head group), blockIdx.y = split: tiles from
// y * per_split on.  The result of a sequence that fits one split goes to `out`,
// else the sums and (m, s) of each head to part [x, splits, 16, DV] and
// ms [x, splits, 16, 2].
// NEW: q, k and v of the newest token come from `fresh`.
template <int D, int DV, typename CT, bool EXT, bool NEW = false>
__global__ __launch_bounds__(256)
void paged_decode_kernel(const short* __restrict__ q,    // [B, Hq, D]
                         const CT* __restrict__ kc,      // [P, 16, Hkv, D]
                         const CT* __restrict__ vc,      // [P, Hkv, DV, 16]
                         const int* __restrict__ bt,     // [B, maxP]
                         const int* __restrict__ seq_lens,
                         short* __restrict__ out,        // [B, Hq, DV]
                         float* __restrict__ part, float* __restrict__ ms,
                         int Hq, int Hkv, int maxP, int Gq, int per_split, int splits,
                         float scale, DecodeExt ext,
                         std::conditional_t<NEW, QkvRope, NoToken> fresh) {
  static_assert(!NEW || (!EXT && D == DV));
  constexpr int NC = D / 32, NT = DV / 16;
  constexpr bool FP8 = sizeof(CT) == 1;
  const int unit = EXT ? blockIdx.x / ext.gchunks : blockIdx.x;
  const int gc = EXT ? blockIdx.x % ext.gchunks : 0;
  const int b = unit / Hkv, kvh = unit % Hkv;
  const int G = EXT ? min(16, Gq - 16 * gc) : Gq;   // heads of this workgroup
  const int L = seq_lens[b];
  const TileRange tr = tile_range<EXT>(L, ext);
  // a length past its page table (whose last page is then read again) may have more
  // tiles than the splits were made for: the last takes them
  const int it0 = blockIdx.y * per_split;
  const int it1 = (int)blockIdx.y + 1 == splits ? tr.n : min(tr.n, it0 + per_split);
  if (blockIdx.y > 0 && it0 >= tr.n) return;
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int hi = lane >> 4, lo = lane & 15;
  const int h0 = kvh * Gq + 16 * gc;
  const int* btb = bt + (long)b * maxP;

  // Q^T fragment: lane holds Q[g = lo][32c + 8hi + j], zero from G on; e4m3 on
  // an fp8 cache, whose bytes feed the MFMA directly
  bf16x8k qf[NC];
  long qf8[NC];
  static_assert(!NEW || (alignof(NewToken<D, CT>) >= 16 && D % 16 == 0));
  __shared__ std::conditional_t<NEW, NewToken<D, CT>, NoToken> now;
  auto take_q = [&] {
#pragma unroll
    for (int c = 0; c < NC; c++) {
      s16x8 raw{};
      if (lo < G) {
        if constexpr (NEW) raw = *reinterpret_cast<const s16x8*>(&now.q[lo][32 * c + 8 * hi]);
        else
          raw = *reinterpret_cast<const s16x8*>(q + ((long)b * Hq + h0 + lo) * D + 32 * c + 8 * hi);
      }
      qf[c] = *reinterpret_cast<bf16x8k*>(&raw);
      if (FP8) {
        float f[8];
#pragma unroll
        for (int j = 0; j < 8; j++) f[j] = bf2f(raw[j]);
        qf8[c] = pack8_fp8(f);
      }
    }
  };
  if constexpr (!NEW) take_q();       // asked for before the pages: 1 x 40 tokens 5.6 us, 6.05 after

  constexpr int LD = DV + 4;               // rows of 16 lanes start at different banks
  __shared__ float Lm[4][16], Ls[4][16];   // per-wave (m, s) of each head
  __shared__ __attribute__((aligned(16))) float Lacc[4][16 * LD];      // per-wave sums

  float m = -INFINITY, sum = 0.f;          // log2 units; of head lo
  f32x4 acc[NT];                           // O^T: rows d = 16t + 4hi + r, column lo
#pragma unroll
  for (int t = 0; t < NT; t++) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  const float sl2 = scale * 1.4426950408889634f;

  auto tile_of = [&](int it) { return it < tr.kept ? it : it - tr.kept + tr.win_tile; };
  auto page = [&](int it, int n) {
    return btb[min(2 * tile_of(min(it, it1 - 1)) + n, maxP - 1)];
  };
  int it = it0 + wid;
  KTile<D, CT> kt;
  int p0 = 0, p1 = 0, p0n = 0, p1n = 0;
  if (it < it1) {
    p0 = page(it, 0);
    p1 = page(it, 1);
    p0n = page(it + 4, 0);
    p1n = page(it + 4, 1);
    kt.load(kc, p0, p1, Hkv, kvh, lo, hi);
  }
  if constexpr (NEW) {
    if ((int)threadIdx.x < (G + 2) * (D / 16))
      now.make(fresh, b, kvh, G, threadIdx.x, blockIdx.y == 0);
    __syncthreads();
    take_q();
  }

  for (; it < it1; it += 4) {
    const int t0 = tile_of(it) * 32;
    // V^T fragments: row d = 16t + lo, tokens 8hi .. + 7 of the two pages
    const CT* vp = vc + (((long)(hi < 2 ? p0 : p1) * Hkv + kvh) * DV + lo) * 16 + 8 * (hi & 1);
    i32x4k v[NT];
#pragma unroll
    for (int t = 0; t < NT; t++) {
      if constexpr (FP8) {
        const i32x2k w = *reinterpret_cast<const i32x2k*>(vp + 256 * t);
        v[t] = i32x4k{w[0], w[1], 0, 0};
      } else {
        v[t] = *reinterpret_cast<const i32x4k*>(vp + 256 * t);
      }
    }
    if constexpr (NEW) {
      // The newest token's place in the tiles that have its page: the last one or, of a length past
      // its table, all that read the table's last page again, where it was put.
      const int own = min((L - 1) >> 4, maxP - 1), at = (L - 1) & 15, first = 2 * tile_of(it);
      if (first + 1 >= own) {
        const bool has[2] = {min(first, maxP - 1) == own, min(first + 1, maxP - 1) == own};
        if (lo == at) {
#pragma unroll
          for (int n = 0; n < 2; n++) {
            if (!has[n]) continue;
#pragma unroll
            for (int c = 0; c < KTile<D, CT>::NV; c++) {
              if constexpr (!FP8) {
                kt.r[n][c] = *reinterpret_cast<const i32x4k*>(&now.k[32 * c + 8 * hi]);
              } else if constexpr (KTile<D, CT>::BYTES >= 16) {
                kt.r[n][c] = *reinterpret_cast<const i32x4k*>(&now.k8[hi * (D / 4) + 16 * c]);
              } else {
                const i32x2k w = *reinterpret_cast<const i32x2k*>(&now.k8[hi * (D / 4)]);
                kt.r[n][c] = i32x4k{w[0], w[1], 0, 0};
              }
            }
          }
        }
        if ((hi < 2 ? has[0] : has[1]) && (hi & 1) == at >> 3) {
          const int bits = FP8 ? 8 * (at & 3) : 16 * (at & 1), word = FP8 ? (at & 7) >> 2
                                                                          : (at & 7) >> 1;
          const unsigned mask = (FP8 ? 0xffu : 0xffffu) << bits;
#pragma unroll
          for (int t = 0; t < NT; t++) {
            unsigned x;
            if constexpr (FP8) x = now.v8[16 * t + lo];
            else x = (unsigned short)now.v[16 * t + lo];
#pragma unroll
            for (int w = 0; w < (FP8 ? 2 : 4); w++)
              if (w == word) v[t][w] = (int)(((unsigned)v[t][w] & ~mask) | x << bits);
          }
        }
      }
    }
    f32x4 sc[2];
#pragma unroll
    for (int n = 0; n < 2; n++) {
      sc[n] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int c = 0; c < NC; c++) {
        if constexpr (FP8) {
          const i32x4k w = kt.r[n][c / 2];
          const i32x2k w2 = c & 1 ? i32x2k{w[2], w[3]} : i32x2k{w[0], w[1]};
          sc[n] = mfma16k_fp8(*reinterpret_cast<const long*>(&w2), qf8[c], sc[n]);
        } else {
          sc[n] = mfma16k(*reinterpret_cast<const bf16x8k*>(&kt.r[n][c]), qf[c], sc[n]);
        }
      }
    }
    p0 = p0n;
    p1 = p1n;
    p0n = page(it + 8, 0);
    p1n = page(it + 8, 1);
    kt.load(kc, p0, p1, Hkv, kvh, lo, hi);
    // ---- online softmax of head lo: 8 of the tile's tokens in this lane ------
    float x[8], top = -INFINITY;
#pragma unroll
    for (int i = 0; i < 8; i++) {
      const int ki = t0 + 16 * (i >> 2) + 4 * hi + (i & 3);
      x[i] = (ki < L && (!EXT || ki >= tr.win_lo || ki < ext.keep)) ? sc[i >> 2][i & 3] * sl2
                                                                    : -INFINITY;
      top = fmaxf(top, x[i]);
    }
    top = max_groups(top);
    float alpha = 1.f;
    if (__any(top > m)) {
      const float mn = fmaxf(m, top);
      alpha = m == -INFINITY ? 0.f : exp2f(m - mn);
      m = mn;
#pragma unroll
      for (int t = 0; t < NT; t++) acc[t] *= alpha;
    }
    const float mm = m == -INFINITY ? 0.f : m;
    float rs = 0.f;
#pragma unroll
    for (int i = 0; i < 8; i++) {
      x[i] = exp2f(x[i] - mm);
      rs += x[i];
    }
    sum = sum * alpha + sum_groups(rs);
    // ---- O^T += V^T P^T ----------------------------------------------------
    if constexpr (FP8) {
      unsigned a = __builtin_amdgcn_cvt_pk_fp8_f32(x[0], x[1], 0, false);
      a = __builtin_amdgcn_cvt_pk_fp8_f32(x[2], x[3], a, true);
      unsigned c = __builtin_amdgcn_cvt_pk_fp8_f32(x[4], x[5], 0, false);
      c = __builtin_amdgcn_cvt_pk_fp8_f32(x[6], x[7], c, true);
      tokens_to_k(a, c);
      const i32x2k w{(int)a, (int)c};
#pragma unroll
      for (int t = 0; t < NT; t++) {
        const i32x2k vv{v[t][0], v[t][1]};
        acc[t] = mfma16k_fp8(*reinterpret_cast<const long*>(&vv),
                             *reinterpret_cast<const long*>(&w), acc[t]);
      }
    } else {
      unsigned w[4];
#pragma unroll
      for (int i = 0; i < 4; i++)
        w[i] = (unsigned)(unsigned short)f2bf(x[2 * i]) |
               (unsigned)(unsigned short)f2bf(x[2 * i + 1]) << 16;
      tokens_to_k(w[0], w[2]);
      tokens_to_k(w[1], w[3]);
      const i32x4k pw{(int)w[0], (int)w[1], (int)w[2], (int)w[3]};
#pragma unroll
      for (int t = 0; t < NT; t++)
        acc[t] = mfma16k(*reinterpret_cast<const bf16x8k*>(&v[t]),
                         *reinterpret_cast<const bf16x8k*>(&pw), acc[t]);
    }
  }

  // ---- cross-wave merge through LDS -----------------------------------
  if (hi == 0) { Lm[wid][lo] = m; Ls[wid][lo] = sum; }
#pragma unroll
  for (int t = 0; t < NT; t++)
    *reinterpret_cast<f32x4*>(&Lacc[wid][lo * LD + 16 * t + 4 * hi]) = acc[t];
  __syncthreads();
  for (int i = threadIdx.x; i < G * (DV / 2); i += 256) {
    const int g = i / (DV / 2), d = 2 * (i % (DV / 2));
    const float M = fmaxf(fmaxf(Lm[0][g], Lm[1][g]), fmaxf(Lm[2][g], Lm[3][g]));
    const float Mf = M == -INFINITY ? 0.f : M;
    float S = 0.f, o0 = 0.f, o1 = 0.f;
#pragma unroll
    for (int w = 0; w < 4; w++) {
      const float c = exp2f(Lm[w][g] - Mf);
      S += Ls[w][g] * c;
      o0 += Lacc[w][g * LD + d] * c;
      o1 += Lacc[w][g * LD + d + 1] * c;
    }
    if (splits == 1 || tr.n <= per_split) {      // nothing to merge
      const float inv = S > 0.f ? 1.f / S : 0.f;
      write_pair<EXT>(out, o0 * inv, o1 * inv, b, h0 + g, d, Hq, DV, ext);
    } else {
      const long row = ((long)blockIdx.x * splits + blockIdx.y) * 16 + g;
      *reinterpret_cast<float2*>(part + row * DV + d) = make_float2(o0, o1);
      if (d == 0) *reinterpret_cast<float2*>(ms + row * 2) = make_float2(M, S);
    }
  }
}

// One wave per (sequence, kv head, head group, head): the splits' sums into out.  A chain of
// latencies: length, maxima, sums.  Up to MOST splits everything is asked for at once, whether
// the sequence has that many or not (what it has not is whatever the memory held): 32 x 2000
// tokens, 12 heads over 2, 17.4 us with the splits one after the other, 15.9.
template <int DV, bool EXT, int MOST>
__global__ __launch_bounds__(64)
void paged_decode_merge_kernel(const float* __restrict__ part, const float* __restrict__ ms,
                               const int* __restrict__ seq_lens, short* __restrict__ out, int Hq,
                               int Hkv, int Gq, int per_split, int splits, DecodeExt ext) {
  const int x = blockIdx.x, g = blockIdx.y;
  const int unit = EXT ? x / ext.gchunks : x, gc = EXT ? x % ext.gchunks : 0;
  const int b = unit / Hkv, kvh = unit % Hkv;
  if (16 * gc + g >= Gq) return;
  const long row0 = (long)x * splits * 16 + g;
  const int lane = threadIdx.x;
  constexpr int NP = DV > 128 ? 2 : 1;      // pairs per lane
  float S = 0.f, o[NP][2] = {};
  if constexpr (MOST > 0) {
    const int len = seq_lens[b];
    float2 w[MOST], v[MOST][NP];
#pragma unroll
    for (int k = 0; k < MOST; k++) {
      const long row = row0 + 16L * min(k, splits - 1);
      w[k] = *reinterpret_cast<const float2*>(ms + row * 2);
#pragma unroll
      for (int j = 0; j < NP; j++)
        v[k][j] = *reinterpret_cast<const float2*>(part + row * DV + min(2 * (lane + 64 * j), DV - 2));
    }
    // (asked for before the first of them is needed)
#pragma unroll
    for (int k = 0; k < MOST; k++) {
      asm volatile("" : "+v"(w[k].x), "+v"(w[k].y));
#pragma unroll
      for (int j = 0; j < NP; j++) asm volatile("" : "+v"(v[k][j].x), "+v"(v[k][j].y));
    }
    const int n = min((tile_range<EXT>(len, ext).n + per_split - 1) / per_split, splits);
    if (n <= 1) return;
    float M = -INFINITY;
#pragma unroll
    for (int k = 0; k < MOST; k++) M = k < n ? fmaxf(M, w[k].x) : M;
    if (M == -INFINITY) M = 0.f;
#pragma unroll
    for (int k = 0; k < MOST; k++) {
      if (k >= n) break;
      const float c = exp2f(w[k].x - M);
      S += w[k].y * c;
#pragma unroll
      for (int j = 0; j < NP; j++) {
        o[j][0] += v[k][j].x * c;
        o[j][1] += v[k][j].y * c;
      }
    }
  } else {
    const int n = min((tile_range<EXT>(seq_lens[b], ext).n + per_split - 1) / per_split, splits);
    if (n <= 1) return;
    float M = -INFINITY;
    for (int k = lane; k < n; k += 64) M = fmaxf(M, ms[(row0 + 16L * k) * 2]);
    M = wave_max(M);
    if (M == -INFINITY) M = 0.f;
#pragma unroll 8
    for (int k = 0; k < n; k++) {
      const long row = row0 + 16L * k;
      const float c = exp2f(ms[row * 2] - M);
      S += ms[row * 2 + 1] * c;
#pragma unroll
      for (int j = 0; j < NP; j++) {
        const int d = 2 * (lane + 64 * j);
        if (d < DV) {
          o[j][0] += part[row * DV + d] * c;
          o[j][1] += part[row * DV + d + 1] * c;
        }
      }
    }
  }
  const float inv = S > 0.f ? 1.f / S : 0.f;
#pragma unroll
  for (int j = 0; j < NP; j++) {
    const int d = 2 * (lane + 64 * j);
    if (d < DV)
      write_pair<EXT>(out, o[j][0] * inv, o[j][1] * inv, b, kvh * Gq + 16 * gc + g, d, Hq, DV, ext);
  }
}

// How a batch of `units` workgroups with at most `tiles` tiles each is split:
// until there is about one per CU, each with at least two tiles for every wave.  Four
// per sequence read 32 x 2000 tokens (12 heads over 2, bf16) in 15.9 us with the
// merge, and, with a merge that took 1.5 more, 17.4, two in 22.5, eight in 22.4 (the first tile's page, key and value
// latencies then outweigh the rest); unsplit it took 135.  At 256 sequences and
// more nothing is split: 2048 x 850 in fp8 take 169 us, 5.3 TB/s.  Nor is a short
// context, whose walk costs no more than the merge (in fp8: 64 x 170 tokens, 9
// tiles, 5.6 us against 7.5, 8 x 400, 19 tiles, 7.1 against 7.5; from 21 tiles on in
// bf16 9.5 against 8.5), nor a batch of which
// part would get a second workgroup per CU (100 x 600: 10.3 against 13.2).
constexpr long DECODE_FILL = 256, UNSPLIT = 20;
struct Splits { int n, per; torch::Tensor part, ms; };
static Splits decode_splits(long units, long tiles, int DV, const torch::Tensor& like) {
  Splits s{1, (int)std::max(tiles, 1L), {}, {}};
  const long want = tiles > UNSPLIT ? std::min((DECODE_FILL + units / 2) / units, (tiles + 7) / 8)
                                    : 1;
  if (want > 1) {
    s.per = (int)((tiles + want - 1) / want + 3) / 4 * 4;
    s.n = (int)((tiles + s.per - 1) / s.per);
  }
  if (s.n > 1) {
    auto f32 = like.options().dtype(torch::kFloat32);
    s.part = torch::empty({units * s.n * 16, (long)DV}, f32);
    s.ms = torch::empty({units * s.n * 16, 2L}, f32);
  }
  return s;
}

template <int DV, bool EXT>
static void launch_merge(dim3 grid, const Splits& sp, const torch::Tensor& seq_lens,
                         torch::Tensor& out, int Hq, int Hkv, int Gq, const DecodeExt& ext) {
#define MERGE(MOST)                                                                          \
  hipLaunchKernelGGL((paged_decode_merge_kernel<DV, EXT, MOST>), grid, dim3(64), 0,          \
                     at::hip::getCurrentHIPStream(), sp.part.data_ptr<float>(),              \
                     sp.ms.data_ptr<float>(), seq_lens.data_ptr<int>(), (short*)out.data_ptr(), \
                     Hq, Hkv, Gq, sp.per, sp.n, ext)
  if (sp.n <= 4) MERGE(4);
  else if (sp.n <= 8) MERGE(8);
  else MERGE(0);
#undef MERGE
}

torch::Tensor paged_attn_decode(torch::Tensor q, torch::Tensor k_cache,
                                torch::Tensor v_cache, torch::Tensor block_tables,
                                torch::Tensor seq_lens, double scale) {
  on_gpu({q, k_cache, v_cache, block_tables, seq_lens});
  TORCH_CHECK(q.scalar_type() == torch::kBFloat16 && q.is_contiguous());
  TORCH_CHECK(block_tables.scalar_type() == torch::kInt && seq_lens.scalar_type() == torch::kInt);
  const int B = q.size(0);
  const int Hq = q.size(1);
  const int D = q.size(2);
  const int page_size = k_cache.size(1);
  const int Hkv = k_cache.size(2);
  const int maxP = block_tables.size(1);
  const int G = Hq / Hkv;
  TORCH_CHECK(page_size == 16, "decode kernel requires page_size == 16");
  TORCH_CHECK(Hq % Hkv == 0 && G <= 16, "GQA group size must be <= 16");
  auto out = torch::empty_like(q);
  if (B == 0) return out;
  auto stream = at::hip::getCurrentHIPStream();
  const Splits sp = decode_splits((long)B * Hkv, (maxP + 1) / 2, D, q);
  float* part = sp.n > 1 ? sp.part.data_ptr<float>() : nullptr;
  float* ms = sp.n > 1 ? sp.ms.data_ptr<float>() : nullptr;
  dim3 grid(B * Hkv, sp.n), block(256);
  const bool fp8 = k_cache.scalar_type() == torch::kFloat8_e4m3fn;
  TORCH_CHECK(fp8 || k_cache.scalar_type() == torch::kBFloat16,
              "kv cache must be bf16 or fp8_e4m3fn");
#define LAUNCH_D(DD, CT)                                                        \
  do {                                                                          \
    hipLaunchKernelGGL((paged_decode_kernel<DD, DD, CT, false>), grid, block, 0, stream, \
                       (const short*)q.data_ptr(), (const CT*)k_cache.data_ptr(), \
                       (const CT*)v_cache.data_ptr(), block_tables.data_ptr<int>(), \
                       seq_lens.data_ptr<int>(), (short*)out.data_ptr(), part, ms, \
                       Hq, Hkv, maxP, G, sp.per, sp.n, (float)scale, DecodeExt{}, NoToken{}); \
    if (sp.n > 1)                                                               \
      launch_merge<DD, false>(dim3(B * Hkv, G), sp, seq_lens, out, Hq, Hkv, G, DecodeExt{}); \
  } while (0)
  if (D == 128) { if (fp8) LAUNCH_D(128, unsigned char); else LAUNCH_D(128, short); }
  else if (D == 64) { if (fp8) LAUNCH_D(64, unsigned char); else LAUNCH_D(64, short); }
  else if (D == 32) { if (fp8) LAUNCH_D(32, unsigned char); else LAUNCH_D(32, short); }
  else { TORCH_CHECK(false, "unsupported head_dim ", D); }
#undef LAUNCH_D
  HIP_CHECK_LAST();
  return out;
}

// qkv_rope_append and paged_attn_decode of what it returns, in one launch: qkv is a decode
// step's projection [B, (Hq + 2 Hkv) D], or its parts and bias; `slots` is where each
// sequence's last position lies.
torch::Tensor paged_attn_decode_new(torch::Tensor qkv, torch::Tensor table, torch::Tensor positions,
                                    torch::Tensor slots, torch::Tensor k_cache,
                                    torch::Tensor v_cache, torch::Tensor block_tables,
                                    torch::Tensor seq_lens, long Hq,
                                    c10::optional<torch::Tensor> bias, double scale) {
  on_gpu({qkv, table, positions, slots, k_cache, v_cache, block_tables, seq_lens, bias});
  check_qkv(qkv, table, positions, slots, k_cache, v_cache, Hq, bias);
  TORCH_CHECK(block_tables.scalar_type() == torch::kInt && seq_lens.scalar_type() == torch::kInt &&
              block_tables.is_contiguous() && seq_lens.is_contiguous());
  const long B = qkv.size(-2), N = qkv.size(-1), Hkv = k_cache.size(2), D = k_cache.size(3);
  const int maxP = block_tables.size(1), G = Hq / Hkv;
  TORCH_CHECK(block_tables.dim() == 2 && block_tables.size(0) == B && seq_lens.numel() == B);
  TORCH_CHECK(k_cache.size(1) == 16, "decode kernel requires page_size == 16");
  TORCH_CHECK(Hq % Hkv == 0 && G <= 16, "GQA group size must be <= 16");
  TORCH_CHECK(D == 32 || D == 64 || D == 128, "unsupported head_dim ", D);
  if ((uintptr_t)qkv.data_ptr() % 16) qkv = qkv.clone();
  if (bias && (uintptr_t)bias->data_ptr() % 16) bias = bias->clone();
  auto out = torch::empty({B, Hq, D}, qkv.options().dtype(torch::kBFloat16));
  if (B == 0) return out;
  QkvRope a{};
  if (qkv.dim() == 3) {
    a.parts = qkv.data_ptr<float>();
    a.part = B * N;
    a.splits = qkv.size(0);
    a.bias = bias ? (const short*)bias->data_ptr() : nullptr;
  } else {
    a.qkv = (const short*)qkv.data_ptr();
  }
  a.table = table.data_ptr<float>();
  a.pos = positions.data_ptr<long>();
  a.slots = slots.data_ptr<long>();
  a.kc = k_cache.data_ptr();
  a.vc = v_cache.data_ptr();
  a.Hq = Hq;
  a.Hkv = Hkv;
  auto stream = at::hip::getCurrentHIPStream();
  const Splits sp = decode_splits(B * Hkv, (maxP + 1) / 2, D, out);
  float* part = sp.n > 1 ? sp.part.data_ptr<float>() : nullptr;
  float* ms = sp.n > 1 ? sp.ms.data_ptr<float>() : nullptr;
#define LAUNCH_N(DD, CT)                                                                       \
  do {                                                                                         \
    hipLaunchKernelGGL((paged_decode_kernel<DD, DD, CT, false, true>), dim3(B * Hkv, sp.n),    \
                       dim3(256), 0, stream, nullptr, (const CT*)k_cache.data_ptr(),           \
                       (const CT*)v_cache.data_ptr(), block_tables.data_ptr<int>(),            \
                       seq_lens.data_ptr<int>(), (short*)out.data_ptr(), part, ms, (int)Hq,    \
                       (int)Hkv, maxP, G, sp.per, sp.n, (float)scale, DecodeExt{}, a);         \
    if (sp.n > 1)                                                                              \
      launch_merge<DD, false>(dim3(B * Hkv, G), sp, seq_lens, out, Hq, Hkv, G, DecodeExt{}); \
  } while (0)
  const bool fp8 = k_cache.scalar_type() == torch::kFloat8_e4m3fn;
  if (D == 128) { if (fp8) LAUNCH_N(128, unsigned char); else LAUNCH_N(128, short); }
  else if (D == 64) { if (fp8) LAUNCH_N(64, unsigned char); else LAUNCH_N(64, short); }
  else { if (fp8) LAUNCH_N(32, unsigned char); else LAUNCH_N(32, short); }
#undef LAUNCH_N
  HIP_CHECK_LAST();
  return out;
}

// General form: key and value widths differ, sliding window with kept first
// tokens, output turned back by position, strided output rows.
// q [B, Hq, DK], k_cache [P, 16, Hkv, DK], v_cache [P, Hkv, DV, 16] (bf16),
// out [B, Hq * V] with any row stride; DK, DV in {32, 64, 128, 256}.
void paged_attn_decode_window(torch::Tensor q, torch::Tensor k_cache, torch::Tensor v_cache,
                              torch::Tensor block_tables, torch::Tensor seq_lens,
                              torch::Tensor out, double scale, long size, long keep,
                              c10::optional<torch::Tensor> uncs) {
  on_gpu({q, k_cache, v_cache, block_tables, seq_lens, out, uncs});
  TORCH_CHECK(q.scalar_type() == torch::kBFloat16 && q.is_contiguous() && q.dim() == 3);
  TORCH_CHECK(k_cache.scalar_type() == torch::kBFloat16 && v_cache.scalar_type() == torch::kBFloat16 &&
              k_cache.is_contiguous() && v_cache.is_contiguous());
  TORCH_CHECK(block_tables.scalar_type() == torch::kInt && block_tables.is_contiguous() &&
              seq_lens.scalar_type() == torch::kInt && seq_lens.is_contiguous());
  const int B = q.size(0), Hq = q.size(1), DK = q.size(2);
  const int Hkv = k_cache.size(2), DV = v_cache.size(2), maxP = block_tables.size(1);
  TORCH_CHECK(k_cache.size(1) == 16 && v_cache.size(3) == 16, "page_size must be 16");
  TORCH_CHECK(k_cache.size(3) == DK && v_cache.size(1) == Hkv && v_cache.size(0) == k_cache.size(0));
  TORCH_CHECK(Hq % Hkv == 0 && block_tables.size(0) == B && seq_lens.numel() == B);
  TORCH_CHECK(out.scalar_type() == torch::kBFloat16 && out.size(0) == B && out.stride(1) == 1 &&
              out.size(1) % Hq == 0);
  TORCH_CHECK(size > 0 && keep >= 0);
  const int V = out.size(1) / Hq;
  TORCH_CHECK(V <= DV);
  if (uncs.has_value())
    TORCH_CHECK(uncs->scalar_type() == torch::kFloat32 && uncs->is_contiguous() &&
                uncs->size(0) == B && uncs->size(1) == V && V % 2 == 0);
  if (B == 0) return;
  const int G = Hq / Hkv;
  DecodeExt e{(int)std::min<long>(size, 1 << 30), (int)std::min<long>(keep, 1 << 30), V,
              out.stride(0), uncs.has_value() ? uncs->data_ptr<float>() : nullptr, (G + 15) / 16};
  auto stream = at::hip::getCurrentHIPStream();
  const long units = (long)B * Hkv * e.gchunks;
  // at most: the whole context, or the window and the kept tokens with their ends
  const long tiles = std::min<long>((maxP + 1) / 2, ((long)e.size + e.keep + 31) / 32 + 2);
  const Splits sp = decode_splits(units, tiles, DV, q);
  float* part = sp.n > 1 ? sp.part.data_ptr<float>() : nullptr;
  float* ms = sp.n > 1 ? sp.ms.data_ptr<float>() : nullptr;
  dim3 grid(units, sp.n), block(256);
#define LAUNCH_KV(KK, VV)                                                                  \
  do {                                                                                     \
    hipLaunchKernelGGL((paged_decode_kernel<KK, VV, short, true>), grid, block, 0, stream, \
                       (const short*)q.data_ptr(), (const short*)k_cache.data_ptr(),       \
                       (const short*)v_cache.data_ptr(), block_tables.data_ptr<int>(),     \
                       seq_lens.data_ptr<int>(), (short*)out.data_ptr(), part, ms, Hq, Hkv, \
                       maxP, G, sp.per, sp.n, (float)scale, e, NoToken{});                 \
    if (sp.n > 1)                                                                          \
      launch_merge<VV, true>(dim3(units, std::min(G, 16)), sp, seq_lens, out, Hq, Hkv, G, e); \
  } while (0)
#define LAUNCH_V(KK)                                                                       \
  do {                                                                                     \
    if (DV == 32) LAUNCH_KV(KK, 32);                                                       \
    else if (DV == 64) LAUNCH_KV(KK, 64);                                                  \
    else if (DV == 128) LAUNCH_KV(KK, 128);                                                \
    else if (DV == 256) LAUNCH_KV(KK, 256);                                                \
    else TORCH_CHECK(false, "unsupported value width ", DV);                               \
  } while (0)
  if (DK == 32) LAUNCH_V(32);
  else if (DK == 64) LAUNCH_V(64);
  else if (DK == 128) LAUNCH_V(128);
  else if (DK == 256) LAUNCH_V(256);
  else TORCH_CHECK(false, "unsupported key width ", DK);
#undef LAUNCH_V
#undef LAUNCH_KV
  HIP_CHECK_LAST();
}

// ----------------------------------------------------------- copies of pages
// pages[dst[i]] = pages[src[i]] in every tensor, 64 of them per launch; a page is
// contiguous.  What samples of one prompt share is computed for the first alone.
struct PagePools {
  char* base[64];
  long bytes[64];        // of a page, multiples of 16
};

__global__ __launch_bounds__(256)
void copy_pages_kernel(PagePools t, const int* __restrict__ src, const int* __restrict__ dst) {
  const long bytes = t.bytes[blockIdx.y];
  const char* from = t.base[blockIdx.y] + src[blockIdx.x] * bytes;
  char* to = t.base[blockIdx.y] + dst[blockIdx.x] * bytes;
  for (long i = threadIdx.x * 16L; i < bytes; i += 256 * 16)
    *reinterpret_cast<uint4*>(to + i) = *reinterpret_cast<const uint4*>(from + i);
}

void copy_pages(std::vector<torch::Tensor> pools, torch::Tensor src, torch::Tensor dst) {
  on_gpu({src, dst});
  TORCH_CHECK(src.scalar_type() == torch::kInt && dst.scalar_type() == torch::kInt &&
              src.is_contiguous() && dst.is_contiguous() && src.numel() == dst.numel(),
              "copy_pages: int32 page numbers");
  const long n = src.numel();
  if (n == 0) return;
  for (size_t i = 0; i < pools.size(); i += 64) {
    PagePools t;
    const size_t here = std::min<size_t>(64, pools.size() - i);
    for (size_t k = 0; k < here; k++) {
      const auto& p = pools[i + k];
      on_gpu({p});
      t.base[k] = (char*)p.data_ptr();
      t.bytes[k] = p.size(0) ? p.numel() / p.size(0) * p.element_size() : 0;
      TORCH_CHECK(p.is_contiguous() && t.bytes[k] % 16 == 0 && (uintptr_t)t.base[k] % 16 == 0,
                  "copy_pages: contiguous pages of whole 16 bytes");
    }
    hipLaunchKernelGGL(copy_pages_kernel, dim3(n, here), dim3(256), 0,
                       c10::hip::getCurrentHIPStream(), t, src.data_ptr<int>(),
                       dst.data_ptr<int>());
  }
  HIP_CHECK_LAST();
}
