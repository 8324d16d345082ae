// Attention of prompt portions over the paged KV cache (the new tokens' own
// keys and values are already in it), so a portion may start anywhere.
//
// paged_attn_varlen (bf16, MFMA): one 256-thread workgroup per (sequence,
// kv-head, 128 query rows).  A "row" is a (token, query head) pair of the
// kv-head's group, tokens outermost, so grouped heads share every K/V tile and
// a short portion still fills the 32-row MFMA tiles.  Each of the 4 waves owns
// 32 rows; KV walks in 64-token tiles (4 pages) that two LDS buffers receive by
// direct loads while the tile before is computed on.  As in the packed forward
// kernel, QK^T is computed swapped (S^T = K Q^T), which leaves a row's 64 scores
// in one lane pair: online softmax without LDS, weights converted to bf16 in
// place, O^T = V^T P^T.  V pages are d-major, so a V^T fragment (8 tokens of one
// d) is 16 bytes; the keys are read in the order that leaves a lane the scores
// of those 8.
//
// What bounds it: of the portions that fill the chip once, a wave's instructions.  A wave alone on
// its SIMD issues one at a time, whichever unit it is for, so the matrix products of a tile (32)
// are hidden only if what else it takes (some 450 instructions) lies between them: a tile's scores
// are computed under the exponentials of the tile before, an LDS read and six VALU instructions to
// a product, which leaves 1.14 us of 1.38 a tile.  Of more workgroups, products, VALU and LDS reads
// together.  12 heads of 128, one tile after the other / now, us: 128 rows over 8064 keys 175 / 145;
// 2048 tokens, 8 times 178 / 162 over a workspace, over pages of 2 heads 177 / 160; 16384 1062 / 950
// and 862 / 805; a window of 1024 over 8 of 693 to 3380 140 / 130.
//
// It takes registers for a second tile's scores, which heads of 128 have: no more than two
// workgroups fit a CU either way.  Narrower ones have up to six, of which three would be left, and
// are overlapped only where there are no more workgroups than CUs (12 heads of 64, 1500 tokens 32.0
// / 27.8, but 40 sequences of 400 in a window of 100 42.9 / 50.5), or, with one width of 128, twice
// as many (16 heads of 128 and 64, 2000 tokens 50 / 40, 16 times 300 20.7 / 26.9).
//
// The same kernel runs over a workspace (LIN) instead of pages: keys [rows, Hkv,
// DK] and transposed values [Hkv * DV, rows] of whole contexts laid out one
// after the other, each from a multiple of 64 rows.
//
// Mask: position i sees j if j <= i and (i - j < size or j < keep); tiles
// between the kept first tokens and the window are never visited.
//
// paged_attn_plain (bf16 or float): one wave per (token, head), scalar
// products in 32-bit; the float32 mode's attention for portions and decoding.
#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>

#include "common.h"
#include "checks.h"

typedef __bf16 bf16x8p __attribute__((ext_vector_type(8)));

DEVINL f32x16 mfma32p(bf16x8p a, bf16x8p b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

struct VarlenArgs {
  const short* q;        // [T, Hq, DK], row stride ldq
  const short* kc;       // [P, 16, Hkv, DK]
  const short* vc;       // [P, Hkv, DV, 16]
  const int* cu;         // [B + 1] first query token of each sequence
  const int* seq_lens;   // [B] keys, the portion's own included
  const int* bt;         // [B, maxP]
  const float* uncs;     // [T, V] cos | sin or null
  short* out;            // [T, ldo], head h at columns h * V
  long ldo, ldq;
  const int* first;      // LIN: first workspace row of each sequence
  long ldv;              // LIN: row stride of vc
  int Hq, Hkv, maxP, V, size, keep;
  int B, tiles;          // sequences, tiles of 128 rows of the longest portion
  float scale;
};

// ---- LDS tiles: rows of 16-byte chunks, the chunks exchanged (xor) by row so
// that 16 rows' reads of one chunk touch every bank once.  V: [d][64 tokens] from
// a workspace; from pages [page][d][16 tokens], as they lie.
template <int D>
DEVINL int row_swz(int row) {
  return D >= 128 ? row & 15 : D == 64 ? (row >> 1) & 7 : (row >> 2) & 3;
}
DEVINL int half_swz(int d) { return (d >> 3) & 1; }

#define INLINE __attribute__((always_inline))

// From so many tiles on a tile's scores are computed under the exponentials of the one before:
// of fewer, what that takes to start outweighs it (64 sequences of 200 tokens, 12 heads over 2 of
// 128, 40.7 us, overlapped 43.2; 16 of 300 31.2 and 31.0).
constexpr int OVERLAPPED = 6;

DEVINL float other_half(float x, int hi) {
  auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(hi ? r[0] : r[1]);
}

template <int DK, int DV, bool LIN, bool PIPE>
__global__ __launch_bounds__(256, (DK > 128 || DV > 128) ? 1 : 2)
void paged_varlen_kernel(VarlenArgs a) {
  constexpr int NDS = DK / 16, NDT = DV / 32, KV = 64;
  constexpr float THR = 11.54f;                // defer-max threshold (log2 units)
  constexpr bool PAIRS = DK <= 128 && DV <= 128;   // two workgroups fit a CU
  int seq, kvh, tile;
  {
    // From 8 kv heads on, a chiplet takes whole heads, whose keys then stay in its
    // L2, long and short rows in turn; else the longest rows first.
    const int n = gridDim.x;
    int id = blockIdx.x;
    if (a.Hkv >= 8) {
      const int q = n >> 3, r = n & 7, xcd = id & 7, mine = id >> 3, all = q + (xcd < r);
      const int first = xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q;
      if (PAIRS && a.B == 1 && n > 256 && n <= 512 && a.size >= a.seq_lens[0]) {
        // One sequence without a window, whose workgroups are more than the CUs, but at most
        // twice as many: some CUs run two, which are the first that a chiplet is given and
        // those after its 32nd.  These are the shortest rows, the longest of them with the
        // shortest and so on; those that are longer, alone, come first among the others.  2708
        // rows of 12 heads after 0, 2708 and 5416 (264 workgroups): 60, 115 and 165 us; long and
        // short in turn 65, 134 and 195.  1500 rows of 40 heads over 8 (472): 50 us, and
        // with two neighbours in length on such a CU 57, long and short in turn 51.
        const int over = max(all - 32, 0);
        int rank = mine < over ? 2 * over - 1 - mine
                   : mine >= 32 ? mine - 32 : 2 * over + (all - over - 1 - mine);
        for (tile = 0;; tile++) {    // the rank'th shortest: a tile's heads are `tiles` ids apart
          const int off = (tile - first % a.tiles + a.tiles) % a.tiles;
          const int same = all / a.tiles + (off < all % a.tiles);
          if (rank < same) {
            id = first + off + rank * a.tiles;
            break;
          }
          rank -= same;
        }
      } else {
        id = first + mine;
        const int t = id % a.tiles;
        tile = t & 1 ? t >> 1 : a.tiles - 1 - (t >> 1);
      }
    } else {
      tile = a.tiles - 1 - id % a.tiles;
    }
    seq = id / a.tiles % a.B;
    kvh = id / a.tiles / a.B;
  }
  const int G = a.Hq / a.Hkv;
  const int t0 = a.cu[seq], nq = a.cu[seq + 1] - t0;
  const int L = a.seq_lens[seq];
  const int start = L - nq;                    // position of the portion's first token
  const int R = nq * G;
  const int r0 = tile * 128;
  if (r0 >= R) return;
  const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 31, hi = lane >> 5;
  const int rw0 = r0 + wid * 32;
  const bool wave_active = rw0 < R;
  const int row = min(rw0 + col, R - 1);
  const bool row_ok = rw0 + col < R;
  const int tok = row / G, head = kvh * G + row % G;
  const int qpos = start + tok;

  __shared__ __attribute__((aligned(512))) short Ks[2][KV * DK], Vs[2][KV * DV];

  bf16x8p qf[NDS];
  {
    const short* qr = a.q + (long)(t0 + tok) * a.ldq + (long)head * DK;
#pragma unroll
    for (int ds = 0; ds < NDS; ds++)
      qf[ds] = *reinterpret_cast<const bf16x8p*>(qr + 16 * ds + 8 * hi);
  }

  float m = -INFINITY, sum = 0.f;
  f32x16 acc[NDT];
#pragma unroll
  for (int t = 0; t < NDT; t++) acc[t] = f32x16{};

  // positions covered by the workgroup and by this wave
  const int pos_lo = start + r0 / G;
  const int pos_hi = start + min(r0 + 127, R - 1) / G;
  const int wpos_lo = start + min(rw0, R - 1) / G;
  const int wpos_hi = start + min(rw0 + 31, R - 1) / G;
  const int win_tile = max(0, pos_lo - a.size + 1) / KV;
  const int kept_tiles = min((a.keep + KV - 1) / KV, win_tile);
  const int ntiles = kept_tiles + pos_hi / KV + 1 - win_tile;
  // scalar loads: a vector load would be waited for behind the tiles under way
  typedef const __attribute__((address_space(4))) int* const_ints;
  const const_ints btb = (const_ints)(size_t)(LIN ? nullptr : a.bt + (long)seq * a.maxP);
  const long lin0 = LIN ? a.first[seq] : 0;
  const int last_page = (L - 1) >> 4;
  auto tile_of = [&](int it) { return it < kept_tiles ? it : it - kept_tiles + win_tile; };

  // A wave's 64 chunks of one load are rows of one page (or 8 rows of V^T).  What does not
  // change from tile to tile is prepared, for a wave alone on its SIMD waits for every
  // scalar instruction; pages are looked up a step before they are needed.
  constexpr int NK = KV * DK / 8 / 256, NV = KV * DV / 8 / 256, PER = 64 / (DK / 8);
  const int ldk = a.Hkv * DK;
  const short* kw = a.kc + kvh * DK + (LIN ? (lin0 + wid * PER) * ldk : (long)(wid * PER % 16) * ldk);
  const short* vw = LIN ? a.vc + ((long)kvh * DV + wid * 8) * a.ldv + lin0
                        : a.vc + ((long)kvh * DV + wid * 32 % DV) * 16;
  auto key_page = [&](int tile, int i) INLINE {
    return btb[min(tile * 4 + ((i * 256 / (DK / 8) + wid * PER) >> 4), last_page)];
  };
  auto value_page = [&](int tile, int i) INLINE {
    return btb[min(tile * 4 + (i * 128 + wid * 32) / DV, last_page)];
  };
  int kpage[NK], vpage[NV];             // of the tiles that are asked for next
  auto key_pages = [&](int tile) INLINE {
    if constexpr (!LIN)
#pragma unroll
      for (int i = 0; i < NK; i++) kpage[i] = key_page(tile, i);
  };
  auto value_pages = [&](int tile) INLINE {
    if constexpr (!LIN)
#pragma unroll
      for (int i = 0; i < NV; i++) vpage[i] = value_page(tile, i);
  };
  auto stage_keys = [&](int tile, int buf) INLINE {
    const short* at = kw + (LIN ? (long)tile * KV * ldk : 0);
#pragma unroll
    for (int i = 0; i < NK; i++) {
      const int row0 = i * 256 / (DK / 8) + wid * PER, r = row0 + lane / (DK / 8);
      const int c = (lane % (DK / 8)) ^ row_swz<DK>(r);
      const long off = LIN ? (long)(i * 256 / (DK / 8)) * ldk
                           : ((long)kpage[i] * 16 + i * 256 / (DK / 8) % 16) * ldk;
      load_to_lds16(at + off, (unsigned)((r - row0) * ldk + c * 8) * 2,
                    &Ks[buf][(i * 256 + wid * 64) * 8]);
    }
  };
  auto stage_values = [&](int tile, int buf) INLINE {
#pragma unroll
    for (int i = 0; i < NV; i++) {
      if constexpr (LIN) {
        const int d = wid * 8 + (lane >> 3), c = (lane & 7) ^ row_swz<64>(d);
        load_to_lds16(vw + tile * KV + (long)(i * 32) * a.ldv,
                      (unsigned)((lane >> 3) * a.ldv + c * 8) * 2,
                      &Vs[buf][(i * 256 + wid * 64) * 8]);
      } else {
        const int d0 = (i * 128 + wid * 32) % DV;
        const int d = d0 + (lane >> 1), c = (lane & 1) ^ half_swz(d);
        load_to_lds16(vw + ((long)vpage[i] * a.Hkv * DV + (d0 - wid * 32 % DV)) * 16,
                      (unsigned)((lane >> 1) * 16 + c * 8) * 2,
                      &Vs[buf][(i * 256 + wid * 64) * 8]);
      }
    }
  };
  // Row i of a key fragment is the key with bits 2 and 3 of i exchanged, which
  // leaves lane half `hi` with keys 16 ks + 8 hi + (0 .. 7) in registers 8 ks + ..
  const int krow = (col & 19) | (col & 4) << 1 | (col & 8) >> 1;

  // scores meet scale * log2(e) in the exponent's fma, which needs a positive scale
  const float sl2 = a.scale * 1.4426950408889634f;
  const float mul = sl2 > 0.f ? sl2 : 1.f;
  // does any of this wave's rows see any of the tile?
  auto visible = [&](int kv0) {
    return wave_active && kv0 <= wpos_hi &&
           !(wpos_lo - (kv0 + KV - 1) >= a.size && kv0 >= a.keep);
  };
  // ... and some of every wave's that has rows?  The same for all waves, and so are the barriers
  // that follow from it.
  const int all_lo = start + min(r0 + 96, R - 1) / G, all_hi = start + min(r0 + 31, R - 1) / G;
  auto visible_to_all = [&](int it) {
    const int kv0 = tile_of(it) * KV;
    return kv0 <= all_hi && !(all_lo - (kv0 + KV - 1) >= a.size && kv0 >= a.keep);
  };
  // A fragment's address is that of its tile's first, which two registers keep, with a
  // constant exchanged (xor) into the chunk and another added.
  typedef __attribute__((address_space(3))) const char* lds_bytes;
  typedef __attribute__((address_space(3))) const bf16x8p* lds_frag;
  const unsigned k0 = lds_address(&Ks[0][0]) + krow * 2 * DK + ((hi ^ row_swz<DK>(krow)) << 4);
  const unsigned v0 = lds_address(&Vs[0][0]) +
                      (LIN ? col * 128 + ((hi ^ row_swz<64>(col)) << 4)
                           : col * 32 + ((hi ^ half_swz(col)) << 4));
  constexpr int AHEAD = 2;              // of a product's fragments, read before it starts
  auto key_frag = [&](unsigned at, int buf, int i) INLINE {
    return *(lds_frag)((lds_bytes)(at ^ (i >> 1) << 5) + (buf * KV + (i & 1) * 32) * 2 * DK);
  };
  auto first_keys = [&](int buf, bf16x8p* f) INLINE {
    unsigned at = k0;
    asm volatile("" : "+v"(at));
#pragma unroll
    for (int i = 0; i < 2 * AHEAD; i++) f[i] = key_frag(at, buf, i);
  };
  auto scores = [&](int buf, f32x16* st, const bf16x8p* first) INLINE {
    unsigned at = k0;
    asm volatile("" : "+v"(at));      // the others made anew each time, or they fill registers
    st[0] = st[1] = f32x16{};
#pragma unroll
    for (int i = 0; i < 2 * NDS; i++)
      st[i & 1] = mfma32p(i < 2 * AHEAD ? first[i] : key_frag(at, buf, i), qf[i >> 1], st[i & 1]);
  };
  auto top_of = [&](const f32x16* st) INLINE {
    float top = st[0][0];
#pragma unroll
    for (int i = 1; i < 32; i++) top = fmaxf(top, st[i >> 4][i & 15]);
    return top;
  };
  auto weigh = [&](int buf, const f32x16* st, float alpha) INLINE {
    const float mm = m == -INFINITY ? 0.f : m;  // a row that sees nothing so far
    float rs = 0.f;
    unsigned at = v0;
    asm volatile("" : "+v"(at));
#pragma unroll
    for (int ks = 0; ks < 4; ks++) {
      union { unsigned u[4]; bf16x8p f; } fr;
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const int i = 8 * ks + 2 * j;
        const float x = __builtin_amdgcn_exp2f(fmaf(st[i >> 4][i & 15], mul, -mm));
        const float y = __builtin_amdgcn_exp2f(fmaf(st[i >> 4][(i & 15) + 1], mul, -mm));
        fr.u[j] = pack2bf(x, y);
        // LIN: normed by the sum of the weights as rounded, so that rounding a
        // weight that stands out does not scale the result
        if constexpr (LIN) rs += __uint_as_float(fr.u[j] << 16) + __uint_as_float(fr.u[j] & 0xffff0000u);
        else rs += x + y;
      }
#pragma unroll
      for (int t = 0; t < NDT; t++)
        acc[t] = mfma32p(LIN ? *(lds_frag)((lds_bytes)(at ^ ks << 5) + (buf * DV + t * 32) * 128)
                             : *(lds_frag)((lds_bytes)at + ((buf * 4 + ks) * DV + t * 32) * 32),
                         fr.f, acc[t]);
    }
    sum = sum * alpha + (rs + other_half(rs, hi));
  };

  // V(it) and K(it + 1) have arrived, K(it) and V(it - 1) are read: the next two are asked for
  auto arrive = [&](int it, int buf, bf16x8p* first) INLINE {
    wait_loads<0>();
    __syncthreads();
    first_keys(buf ^ 1, first);
    if (it + 2 < ntiles) stage_keys(tile_of(it + 2), buf);
    if (it + 1 < ntiles) stage_values(tile_of(it + 1), buf ^ 1);
    key_pages(tile_of(it + 3));
    value_pages(tile_of(it + 2));
  };
  // mask and maximum of a tile's scores, of which `top` is a lane's largest; rescales if needed
  auto settle = [&](int kv0, f32x16* st, float top) INLINE {
    if (!(sl2 > 0.f)) {
#pragma unroll
      for (int i = 0; i < 32; i++) st[i >> 4][i & 15] *= sl2;
      top = top_of(st);
    }
    const bool full = kv0 + KV - 1 <= wpos_lo &&
                      (wpos_hi - kv0 < a.size || kv0 + KV <= a.keep);
    if (!full) {
      int see = qpos - kv0 - 8 * hi;                      // counted from the lane's first key
      int kept = a.keep - kv0 - 8 * hi;
      asm volatile("" : "+v"(see), "+v"(kept));
#pragma unroll
      for (int i = 0; i < 32; i++) {
        const int ki = 16 * (i >> 3) + (i & 7);
        if (!(ki <= see && (see - ki < a.size || ki < kept))) st[i >> 4][i & 15] = -INFINITY;
      }
      top = top_of(st);
    }
    const float pmax = fmaxf(top, other_half(top, hi)) * mul;
    float alpha = 1.f;
    if (__any(!(pmax - m <= THR))) {           // also true while m is -inf
      const float mn = fmaxf(m, pmax);
      alpha = (m == -INFINITY) ? 0.f : exp2f(m - mn);
      m = mn;
#pragma unroll
      for (int t = 0; t < NDT; t++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[t][r] *= alpha;
    }
    return alpha;
  };
  // one tile, the next one's scores under its exponentials
  auto both = [&](int it, int buf, f32x16* cur, float top, f32x16* next, float& ntop) INLINE {
    bf16x8p first[2 * AHEAD];
    arrive(it, buf, first);
    if (!wave_active) return;
    const float alpha = settle(tile_of(it) * KV, cur, top);
    __builtin_amdgcn_sched_barrier(0);
    scores(buf ^ 1, next, first);
    weigh(buf, cur, alpha);
    ntop = top_of(next);
    asm volatile("" : "+v"(ntop));
    // a product, six VALU instructions and the read of the product after the next, in turn
    __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
#pragma unroll
    for (int i = 0; i < 2 * NDS + 4 * NDT; i++) {
      __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x402, 6, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  f32x16 s0[2] = {}, s1[2];
  float top0 = 0.f, top1 = 0.f;
  auto one = [&](int it, int buf) INLINE {
    bf16x8p first[2 * AHEAD];
    arrive(it, buf, first);
    const int kv0 = tile_of(it) * KV;
    if (visible(kv0)) weigh(buf, s0, settle(kv0, s0, top0));
    if (it + 1 < ntiles && visible(tile_of(it + 1) * KV)) {
      scores(buf ^ 1, s0, first);
      top0 = top_of(s0);
    }
  };

#pragma unroll
  for (int ds = 0; ds < NDS; ds++) asm volatile("" : "+v"(qf[ds]));   // arrived
  key_pages(tile_of(0));
  value_pages(tile_of(0));
  stage_keys(tile_of(0), 0);
  stage_values(tile_of(0), 0);
  bool piped = false;
  if constexpr (PIPE) piped = ntiles >= OVERLAPPED;
  if (piped) {
    key_pages(tile_of(1));
    wait_loads<NV>();         // the keys
    __syncthreads();
    stage_keys(tile_of(1), 1);
    key_pages(tile_of(2));
    value_pages(tile_of(1));
    if (visible(tile_of(0) * KV)) {
      bf16x8p first[2 * AHEAD];
      first_keys(0, first);
      scores(0, s0, first);
      top0 = top_of(s0);
    }
    for (int it = 0; it < ntiles; it += 2) {
      // (a loop of its own, or the scores change registers in every round)
      for (; it + 2 < ntiles && visible_to_all(it) && visible_to_all(it + 1) &&
             visible_to_all(it + 2); it += 2) {
        both(it, 0, s0, top0, s1, top1);
        both(it + 1, 1, s1, top1, s0, top0);
      }
      one(it, 0);
      if (it + 1 < ntiles) one(it + 1, 1);
    }
  } else {
    for (int it = 0; it < ntiles; it++) {
      const int buf = it & 1, kv0 = tile_of(it) * KV;
      wait_loads<0>();
      __syncthreads();
      if (it + 1 < ntiles) {
        key_pages(tile_of(it + 1));
        value_pages(tile_of(it + 1));
        stage_keys(tile_of(it + 1), buf ^ 1);
        stage_values(tile_of(it + 1), buf ^ 1);
      }
      if (!visible(kv0)) continue;
      bf16x8p first[2 * AHEAD];
      f32x16 st[2];
      first_keys(buf, first);
      scores(buf, st, first);
      weigh(buf, st, settle(kv0, st, top_of(st)));
    }
  }

  if (!wave_active || !row_ok) return;
  const float inv = sum > 0.f ? 1.f / sum : 0.f;
  short* op = a.out + (long)(t0 + tok) * a.ldo + (long)head * a.V;
  const float* cs = a.uncs ? a.uncs + (long)(t0 + tok) * a.V : nullptr;
  const int half = a.V / 2;
  const bool wide = (a.V & 3) == 0 && (a.ldo & 3) == 0 && ((size_t)a.out & 7) == 0;
#pragma unroll
  for (int t = 0; t < NDT; t++)
#pragma unroll
    for (int g = 0; g < 4; g++) {
      const int d0 = t * 32 + 8 * g + 4 * hi;   // registers 4g..4g+3 are d0..d0+3
      if (d0 >= a.V) continue;
      float o[4];
#pragma unroll
      for (int j = 0; j < 4; j++) o[j] = acc[t][4 * g + j] * inv;
      if (cs) {
#pragma unroll
        for (int j = 0; j < 4; j += 2) {
          const int pr = min((d0 + j) >> 1, half - 1);
          const float c = cs[pr], s = cs[half + pr], u = o[j], v = o[j + 1];
          o[j] = u * c + v * s;
          o[j + 1] = v * c - u * s;
        }
      }
      if (wide)
        stv<4>(op + d0, o);
      else
#pragma unroll
        for (int j = 0; j < 4; j++)
          if (d0 + j < a.V) stf(op + d0 + j, o[j]);
    }
}

// -------------------------------------------------------- plain, any type
template <typename T>
__global__ __launch_bounds__(256) void paged_plain_kernel(
    const T* __restrict__ q, const T* __restrict__ kc, const T* __restrict__ vc,
    const int* __restrict__ row_seq, const long* __restrict__ positions,
    const int* __restrict__ bt, const float* __restrict__ uncs, T* __restrict__ out,
    long rows, int Hq, int Hkv, int DK, int DV, int V, int maxP, long ldo, int size, int keep,
    float scale) {
  __shared__ float qs[4][256], ps[4][64], os[4][256];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const long unit = blockIdx.x * 4L + w;
  if (unit >= rows * Hq) return;
  const long t = unit / Hq;
  const int h = (int)(unit % Hq), kvh = h / (Hq / Hkv);
  const int pos = (int)positions[t];
  const int* btb = bt + (long)row_seq[t] * maxP;
  for (int d = lane; d < DK; d += 64) qs[w][d] = ldf(q + (t * Hq + h) * (long)DK + d);
  lds_fence_wave_kv();
  float m = -INFINITY, sum = 0.f, acc[4] = {0.f, 0.f, 0.f, 0.f};
  const int win_tile = max(0, pos - size + 1) / 64;
  const int kept = min((keep + 63) / 64, win_tile);
  const int n = kept + pos / 64 + 1 - win_tile;
  for (int it = 0; it < n; it++) {
    const int k0 = (it < kept ? it : it - kept + win_tile) * 64;
    const int ki = k0 + lane;
    float s = -INFINITY;
    if (ki <= pos && (pos - ki < size || ki < keep)) {
      const T* kr = kc + (((long)btb[min(ki >> 4, maxP - 1)] * 16 + (ki & 15)) * Hkv + kvh) * DK;
      float d0 = 0.f;
      for (int d = 0; d < DK; d += 4) {
        float v[4];
        ldv<4>(kr + d, v);
#pragma unroll
        for (int j = 0; j < 4; j++) d0 += v[j] * qs[w][d + j];
      }
      s = d0 * scale;
    }
    const float mn = fmaxf(m, wave_max(s));
    const float alpha = (m == -INFINITY) ? 0.f : expf(m - mn);
    const float p = (s == -INFINITY) ? 0.f : expf(s - mn);
    m = mn;
    sum = sum * alpha + wave_sum(p);
    ps[w][lane] = p;
    lds_fence_wave_kv();
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int d = lane + 64 * r;
      acc[r] *= alpha;
      if (d >= V) continue;
      for (int pg = 0; pg < 4; pg++) {
        if (k0 + 16 * pg > pos) break;
        const T* vr = vc + (((long)btb[min((k0 >> 4) + pg, maxP - 1)] * Hkv + kvh) * DV + d) * 16;
        for (int j = 0; j < 16; j++) acc[r] += ps[w][16 * pg + j] * ldf(vr + j);
      }
    }
    lds_fence_wave_kv();
  }
#pragma unroll
  for (int r = 0; r < 4; r++)
    if (lane + 64 * r < V) os[w][lane + 64 * r] = acc[r] / sum;
  lds_fence_wave_kv();
  T* op = out + t * ldo + (long)h * V;
  const int half = V / 2;
  for (int d = lane; d < V; d += 64) {
    float o = os[w][d];
    if (uncs) {
      const float c = uncs[t * V + (d >> 1)], s = uncs[t * V + half + (d >> 1)];
      o = o * c + ((d & 1) ? -os[w][d ^ 1] : os[w][d ^ 1]) * s;
    }
    stf(op + d, o);
  }
}

// ======================================================== host wrappers ==
static void check_cache(const torch::Tensor& q, const torch::Tensor& kc, const torch::Tensor& vc,
                        const torch::Tensor& bt, const torch::Tensor& out,
                        const c10::optional<torch::Tensor>& uncs, long size, long keep) {
  on_gpu({q, kc, vc, bt, out, uncs});
  TORCH_CHECK(q.dim() == 3 && q.is_contiguous());
  TORCH_CHECK(kc.is_contiguous() && vc.is_contiguous() && kc.dim() == 4 && vc.dim() == 4);
  TORCH_CHECK(kc.scalar_type() == q.scalar_type() && vc.scalar_type() == q.scalar_type() &&
              out.scalar_type() == q.scalar_type(), "q, cache and output of one type");
  TORCH_CHECK(kc.size(1) == 16 && vc.size(3) == 16, "page_size must be 16");
  TORCH_CHECK(kc.size(3) == q.size(2) && vc.size(1) == kc.size(2) && vc.size(0) == kc.size(0));
  TORCH_CHECK(q.size(1) % kc.size(2) == 0);
  TORCH_CHECK(bt.scalar_type() == torch::kInt && bt.is_contiguous() && bt.dim() == 2 && bt.size(1) > 0);
  TORCH_CHECK(out.dim() == 2 && out.size(0) == q.size(0) && out.stride(1) == 1 &&
              out.size(1) % q.size(1) == 0 && out.size(1) / q.size(1) <= vc.size(2));
  TORCH_CHECK(size > 0 && keep >= 0);
  if (uncs.has_value())
    TORCH_CHECK(uncs->scalar_type() == torch::kFloat32 && uncs->is_contiguous() &&
                uncs->size(0) == q.size(0) && uncs->size(1) * q.size(1) == out.size(1) &&
                uncs->size(1) % 2 == 0);
}

template <bool LIN>
static void launch_varlen(VarlenArgs a, int DK, int DV, long max_rows, hipStream_t stream) {
  a.tiles = (max_rows + 127) / 128;
  if (!a.tiles) return;
  const dim3 grid((unsigned)((long)a.tiles * a.B * a.Hkv));
  const long longest = LIN ? a.ldv : 16L * a.maxP;      // a context, at most
  const bool pipe = longest > 64 * (OVERLAPPED - 1) &&
                    ((DK == 128 && DV == 128) || grid.x <= (DK + DV > 128 ? 512 : 256));
#define LAUNCH(KK, VV)                                                                           \
  do {                                                                                           \
    if (pipe && KK <= 128 && VV <= 128)                                                          \
      hipLaunchKernelGGL((paged_varlen_kernel<KK, VV, LIN, (KK <= 128 && VV <= 128)>), grid,     \
                         dim3(256), 0, stream, a);                                               \
    else                                                                                         \
      hipLaunchKernelGGL((paged_varlen_kernel<KK, VV, LIN, false>), grid, dim3(256), 0, stream, a); \
  } while (0)
#define LAUNCH_V(KK)                                              \
  do {                                                            \
    if (DV == 32) LAUNCH(KK, 32);                                 \
    else if (DV == 64) LAUNCH(KK, 64);                            \
    else if (DV == 128) LAUNCH(KK, 128);                          \
    else if (DV == 256) LAUNCH(KK, 256);                          \
    else TORCH_CHECK(false, "unsupported value width ", DV);      \
  } while (0)
  if (DK == 32) LAUNCH_V(32);
  else if (DK == 64) LAUNCH_V(64);
  else if (DK == 128) LAUNCH_V(128);
  else if (DK == 256) LAUNCH_V(256);
  else TORCH_CHECK(false, "unsupported key width ", DK);
#undef LAUNCH_V
#undef LAUNCH
  HIP_CHECK_LAST();
}

void paged_attn_varlen(torch::Tensor q, torch::Tensor kc, torch::Tensor vc, torch::Tensor cu,
                       torch::Tensor seq_lens, torch::Tensor bt, torch::Tensor out, long max_q,
                       double scale, long size, long keep, c10::optional<torch::Tensor> uncs) {
  check_cache(q, kc, vc, bt, out, uncs, size, keep);
  TORCH_CHECK(q.scalar_type() == torch::kBFloat16);
  const int B = seq_lens.numel();
  on_gpu({cu, seq_lens});
  TORCH_CHECK(cu.scalar_type() == torch::kInt && cu.is_contiguous() && cu.numel() == B + 1 &&
              seq_lens.scalar_type() == torch::kInt && seq_lens.is_contiguous() && bt.size(0) == B);
  if (B == 0 || q.size(0) == 0) return;
  VarlenArgs a;
  a.q = (const short*)q.data_ptr();
  a.kc = (const short*)kc.data_ptr();
  a.vc = (const short*)vc.data_ptr();
  a.cu = cu.data_ptr<int>();
  a.seq_lens = seq_lens.data_ptr<int>();
  a.bt = bt.data_ptr<int>();
  a.uncs = uncs.has_value() ? uncs->data_ptr<float>() : nullptr;
  a.out = (short*)out.data_ptr();
  a.ldo = out.stride(0);
  a.ldq = q.size(1) * q.size(2);
  a.first = nullptr;
  a.ldv = 0;
  a.Hq = q.size(1);
  a.Hkv = kc.size(2);
  a.maxP = bt.size(1);
  a.V = out.size(1) / q.size(1);
  a.size = (int)std::min<long>(size, 1 << 30);
  a.keep = (int)std::min<long>(keep, 1 << 30);
  a.scale = scale;
  const int DK = q.size(2), DV = vc.size(2);
  a.B = B;
  launch_varlen<false>(a, DK, DV, max_q * (a.Hq / a.Hkv), at::hip::getCurrentHIPStream());
}

// Attention of portions over expanded contexts: q [T, Hq * DK] (any row
// stride), k [rows, Hq * DK], vt [Hq * DV, rows]; sequence b's context starts at
// row first[b], a multiple of 64, and first[B] == rows.
void expanded_attn_varlen(torch::Tensor q, torch::Tensor k, torch::Tensor vt, torch::Tensor cu,
                          torch::Tensor seq_lens, torch::Tensor first, torch::Tensor out,
                          long heads, long max_q, double scale) {
  const long B = seq_lens.numel(), rows = k.size(0);
  on_gpu({q, k, vt, cu, seq_lens, first, out});
  for (auto& t : {q, k, vt, out})
    TORCH_CHECK(t.dim() == 2 && t.stride(1) == 1 &&
                t.scalar_type() == torch::kBFloat16);
  TORCH_CHECK(k.is_contiguous() && vt.is_contiguous() && q.size(1) == k.size(1) &&
              k.size(1) % heads == 0 && vt.size(0) % heads == 0 && vt.size(1) == rows &&
              rows % 64 == 0 && out.size(0) == q.size(0) && out.size(1) % heads == 0);
  TORCH_CHECK(q.stride(0) % 8 == 0 && (uintptr_t)q.data_ptr() % 16 == 0);
  for (auto& t : {cu, seq_lens, first})
    TORCH_CHECK(t.scalar_type() == torch::kInt && t.is_contiguous());
  TORCH_CHECK(cu.numel() == B + 1 && first.numel() == B + 1);
  if (B == 0 || q.size(0) == 0) return;
  VarlenArgs a{};
  a.q = (const short*)q.data_ptr();
  a.kc = (const short*)k.data_ptr();
  a.vc = (const short*)vt.data_ptr();
  a.cu = cu.data_ptr<int>();
  a.seq_lens = seq_lens.data_ptr<int>();
  a.first = first.data_ptr<int>();
  a.out = (short*)out.data_ptr();
  a.ldo = out.stride(0);
  a.ldq = q.stride(0);
  a.ldv = rows;
  a.Hq = a.Hkv = heads;
  a.V = out.size(1) / heads;
  a.size = 1 << 30;
  a.scale = scale;
  const int DK = k.size(1) / heads, DV = vt.size(0) / heads;
  TORCH_CHECK(a.V <= DV);
  a.B = B;
  launch_varlen<true>(a, DK, DV, max_q, at::hip::getCurrentHIPStream());
}

void paged_attn_plain(torch::Tensor q, torch::Tensor kc, torch::Tensor vc, torch::Tensor row_seq,
                      torch::Tensor positions, torch::Tensor bt, torch::Tensor out, double scale,
                      long size, long keep, c10::optional<torch::Tensor> uncs) {
  check_cache(q, kc, vc, bt, out, uncs, size, keep);
  const long rows = q.size(0);
  on_gpu({row_seq, positions});
  TORCH_CHECK(row_seq.scalar_type() == torch::kInt && row_seq.is_contiguous() && row_seq.numel() == rows);
  TORCH_CHECK(positions.scalar_type() == torch::kLong && positions.is_contiguous() && positions.numel() == rows);
  const int DK = q.size(2), DV = vc.size(2), V = out.size(1) / q.size(1);
  TORCH_CHECK(DK <= 256 && DV <= 256 && DK % 4 == 0);
  if (rows == 0) return;
  const long units = rows * q.size(1);
  auto stream = at::hip::getCurrentHIPStream();
#define LAUNCH(TT)                                                                            \
  hipLaunchKernelGGL((paged_plain_kernel<TT>), dim3((units + 3) / 4), dim3(256), 0, stream,   \
                     (const TT*)q.data_ptr(), (const TT*)kc.data_ptr(), (const TT*)vc.data_ptr(), \
                     row_seq.data_ptr<int>(), positions.data_ptr<long>(), bt.data_ptr<int>(), \
                     uncs.has_value() ? uncs->data_ptr<float>() : nullptr, (TT*)out.data_ptr(), \
                     rows, (int)q.size(1), (int)kc.size(2), DK, DV, V, (int)bt.size(1),        \
                     out.stride(0), (int)std::min<long>(size, 1 << 30),                        \
                     (int)std::min<long>(keep, 1 << 30), (float)scale)
  if (q.scalar_type() == torch::kBFloat16) LAUNCH(short);
  else {
    TORCH_CHECK(q.scalar_type() == torch::kFloat32);
    LAUNCH(float);
  }
#undef LAUNCH
  HIP_CHECK_LAST();
}
