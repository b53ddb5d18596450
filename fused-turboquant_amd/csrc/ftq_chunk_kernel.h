// Attention of a chunk of consecutive query tokens of one sequence over a
// compressed K/V cache (the continuation of a chunked prefill): causal, every
// query row r attends positions [lo(r), past + r + 1).
//
// The decode kernels dequantise the cache once per (query token, kv head); a
// chunk of n tokens that goes through them as n synthetic sequences
// dequantises it n times.  Here the cache is dequantised once per chunk, into
// the exact operands of the matrix cores (not into rounded K and V), and a
// flash-attention kernel then shares every 64-token tile among 128 (64 at
// D = 256) query columns:
//   gather   codes -> K table values (f16, or f16 hi + lo where the decode
//            kernel of that format keeps fp32 products) and V codes (centred,
//            exact in f16), in MFMA fragment order, plus 4 floats per token:
//            K factor, bias (0, or -inf for a position without a page), V
//            factor, V minimum
//   queries  rotated, scaled by scale * log2 e, f16 hi + lo, fragment order
//   attend   S^T = K Q^T, softmax in the log2 domain, O^T = V^T P^T
//
// Fragment order: lane (m, g) of v_mfma_f32_16x16x32_f16 (m = lane & 15,
// g = lane >> 4) reads 16 contiguous bytes, and a wave 1 KB:
//   K  [16-token tile][32-dim step s][part][lane]: token m, dims 32 s + 8 g + j
//   V  [32-token tile][16-dim block b][part][lane]: dim 16 b + m, tokens 4 g + j and
//      16 + 4 g + j (j < 4) -- the row order of the S^T accumulators, so P goes
//      from the score registers into the P.V operand without a shuffle
//   Q  [16-column tile][s][part][lane]: column m, dims 32 s + 8 g + j
// A column is a (query row, head of the kv head's group) pair, row-major.
//
// Bound by the matrix cores and the softmax beside them: the hi + lo query and
// weights double the products, and 1024 query tokens over 6144 positions (32
// heads over 8 at d = 128, 4-bit) run 189 GFLOP of them in 182 us, 1.04
// PFLOP/s where a large library product in the same type reaches 1.33.  Before
// that: 231 us with the tiles staged through registers and the masks of the
// edges in every tile.  The tiles now go to LDS directly (17 registers free,
// which is what lets the low parts and the sums run under the high parts'
// products), and only the tiles at the edges of the causal range or the window
// carry masks, in a copy of the loop.  d = 64: 190 -> 157 us; d = 256 (8 heads
// over 4): 197 -> 155; d = 128 with 8-bit K and V: 329 -> 223.
#pragma once

#include "ftq_attn_dev.h"
#include "ftq_merge.h"
#include "ftq_v1_dev.h"

#include <type_traits>

namespace ftq {

// Query columns of a workgroup (4 waves) and tokens of a tile.
template <int D, bool KHL> struct ChunkGeo {
  static constexpr int CT = D == 256 ? 1 : 2;     // 16-column tiles per wave
  static constexpr int COLS = 64 * CT;
  static constexpr int TK = D == 64 ? 64 : 32;
  static constexpr int NS = D / 32, NB = D / 16, NT = TK / 16, NP = TK / 32;
};

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

struct ChunkAttn {
  const u32x4 *kf, *vf, *qf;   // fragments: [kv head][...]
  const float* tok;            // [kv head][tile][4][TK]: K factor, bias, V factor, V minimum
  const float* qfac;           // per column factor of the scores ([kv head][column]); KHL and NH == 1
  int64_t kstride, vstride, qstride;  // uint4 per kv head
  int64_t tstride;             // floats per kv head
  int cstride;                 // columns per kv head (qfac)
  int nq, G, hq, hkv, past, window;  // hq, hkv: of all sequences; past: the longest, for the grid
  const int32_t* lens;         // per sequence, past = lens[b] - lens_less; null: one sequence, `past`
  int hkv_b, lens_less;        // kv heads of one sequence
  int seg0, seg1;              // token range held by the fragments (seg0 a multiple of 64)
  int splits, split0, splits_all;  // splits of this launch, its first split, all splits of the row
  float *wo, *wl;              // partial outputs / log-sum-exps, or
  void* out;                   // the output itself (wo == null)
  int ot, rot;                 // output dtype; MergeRot of the direct output (ROT_NONE / PLAIN / SIGNS)
  const float* signs;
  float vscale;                // of the accumulators: undoes the V operands' and factors' common power of two
  float oscale;                // of the un-rotation (direct output only)
  int64_t o_batch, o_row, o_head;  // output strides (elements) of a sequence, a query row and a head
  int nan_zero;                // a row with a NaN score is zeros (decode steps); else NaN
};

// x of the lane 16 (32) lanes up or down: the butterfly pair of lane bit 4 (5)
__device__ __forceinline__ float fwht_pair16(float x, bool upper) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  const float a = __uint_as_float(r[0]), b = __uint_as_float(r[1]);
  return upper ? a - b : a + b;
}
__device__ __forceinline__ float fwht_pair32(float x, bool upper) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  const float a = __uint_as_float(r[0]), b = __uint_as_float(r[1]);
  return upper ? a - b : a + b;
}

// 16 (4) bytes of each lane to base + 16 (4) * lane in LDS; base is the wave's
__device__ __forceinline__ void lds_load16(const void* src, void* base) {
  __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
                                   (__attribute__((address_space(3))) void*)base, 16, 0, 0);
}
__device__ __forceinline__ void lds_load4(const void* src, void* base) {
  __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
                                   (__attribute__((address_space(3))) void*)base, 4, 0, 0);
}

// f16 pair of two floats, each rounded to nearest (v_cvt_pk_f16_f32)
__device__ __forceinline__ uint32_t pk_f16(float a, float b) {
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{a, b}), half2_t));
}
// x - f16 half of w
__device__ __forceinline__ float f16_rest(float x, uint32_t w, int half) {
  return x - (float)__builtin_bit_cast(half2_t, w)[half];
}

// D: head dim; NH: f16 parts of the query and of the weights (2: ~22 bits, as
// the v1 decode kernels; 1: f16); KHL: K fragments as hi + lo and the query
// scaled per column (formats whose decode runs fp32 products); VHL: V
// fragments as hi + lo (Lloyd-Max V at that precision); ZM: V has a per-token
// minimum, and positions may be hidden by their bias.
template <int D, int NH, bool KHL, bool VHL, bool ZM>
__global__ __launch_bounds__(256, D == 256 ? 1 : 2) void chunk_attn_kernel(const ChunkAttn a) {
  using C = ChunkGeo<D, KHL>;
  constexpr int CT = C::CT, TK = C::TK, NS = C::NS, NB = C::NB, NT = C::NT, NP = C::NP;
  constexpr int KP = KHL ? 2 : 1;
  constexpr int VP = VHL ? 2 : 1;
  static_assert(!VHL || KHL, "V hi + lo goes with K hi + lo");
  constexpr int KU = NT * NS * KP * 64, VU = NP * NB * VP * 64;  // 16-byte units of a tile
  static_assert(KU % 256 == 0 && VU % 256 == 0 && 4 * TK % 64 == 0, "whole waves fetch a tile");
  __shared__ u32x4 kb[2][KU];
  __shared__ u32x4 vb[2][VU];
  __shared__ __attribute__((aligned(16))) float tb[2][4][TK];

  // kv head fastest: with 8 kv heads each XCD (workgroups are dealt to the 8
  // XCDs in turn) reads one head's fragments, which then stay in its L2
  const int kvh = blockIdx.x % a.hkv;
  const int blk = (int)(gridDim.x / a.hkv) - 1 - (int)(blockIdx.x / a.hkv);  // longest rows first
  const int split = blockIdx.y;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int n = lane & 15, g = lane >> 4;
  const int ncols = a.nq * a.G;
  const int seq = kvh / a.hkv_b;
  const int past = a.lens != nullptr ? a.lens[seq] - a.lens_less : a.past;

  // the rows of this workgroup, wave and lane
  const int c0 = blk * C::COLS;
  const int r_lo = c0 / a.G, r_hi = (min(c0 + C::COLS, ncols) - 1) / a.G;
  const int wc0 = c0 + wave * 16 * CT;
  const int first = a.window > 0 ? max(0, past + r_lo + 1 - a.window) : 0;
  const int t0 = max(first, a.seg0) / TK;
  const int t1 = (min(past + r_hi + 1, a.seg1) + TK - 1) / TK;
  const int nt = t1 > t0 ? t1 - t0 : 0;
  const int per = (nt + a.splits - 1) / a.splits;
  const int tb0 = t0 + split * per, tb1 = min(tb0 + per, t1);
  // positions that every row of the workgroup attends: [w_from, w_all)
  const int w_all = past + r_lo + 1;
  const int w_from = a.window > 0 ? max(0, past + r_hi + 1 - a.window) : 0;
  int lim[CT], lo[CT];
#pragma unroll
  for (int ct = 0; ct < CT; ++ct) {
    const int r = min((wc0 + 16 * ct + n) / a.G, a.nq - 1);
    lim[ct] = past + r + 1;
    lo[ct] = a.window > 0 ? max(0, lim[ct] - a.window) : 0;
  }

  const u32x4* kf = a.kf + (int64_t)kvh * a.kstride;
  const u32x4* vf = a.vf + (int64_t)kvh * a.vstride;
  const float* tk = a.tok + (int64_t)kvh * a.tstride;
  const int tseg = a.seg0 / TK;
  // a tile's fragments go straight to LDS (fragment order is lane order)
  auto fetch = [&](int t, int p) __attribute__((always_inline)) {
    const u32x4* pk = kf + (int64_t)(t - tseg) * KU + tid;
    const u32x4* pv = vf + (int64_t)(t - tseg) * VU + tid;
#pragma unroll
    for (int j = 0; j < KU / 256; ++j) lds_load16(pk + 256 * j, &kb[p][256 * j + 64 * wave]);
#pragma unroll
    for (int j = 0; j < VU / 256; ++j) lds_load16(pv + 256 * j, &vb[p][256 * j + 64 * wave]);
    if (wave < 4 * TK / 64) lds_load4(tk + (int64_t)(t - tseg) * 4 * TK + tid, &tb[p][0][0] + 64 * wave);
  };

  if (tb0 < tb1) fetch(tb0, 0);
  // the query operands of the wave's columns
  half8 qh[CT][NS], ql[NH == 2 ? CT : 1][NH == 2 ? NS : 1];
  float qs[CT];
  bool qlarge = false;  // NH == 1: a column whose query was scaled to stay an f16 number; rare
#pragma unroll
  for (int ct = 0; ct < CT; ++ct) {
    const u32x4* pq = a.qf + (int64_t)kvh * a.qstride + (int64_t)(wc0 / 16 + ct) * (NS * NH * 64) + lane;
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      qh[ct][s] = __builtin_bit_cast(half8, pq[(s * NH) * 64]);
      if constexpr (NH == 2) ql[ct][s] = __builtin_bit_cast(half8, pq[(s * NH + 1) * 64]);
    }
    qs[ct] = KHL || NH == 1 ? a.qfac[(int64_t)kvh * a.cstride + wc0 + 16 * ct + n] : 1.f;
    if constexpr (!KHL && NH == 1)
      qlarge = qlarge || __builtin_amdgcn_ballot_w64(qs[ct] > 1.f && wc0 + 16 * ct + n < ncols) != 0;  // wave-uniform
  }

  constexpr float TAU = 4.f;        // weights stay below 2^TAU
  constexpr float MINF = -3.0e38f;  // running maximum of a column with no position yet
  float m_run[CT], l_run[CT], z_run[CT];
  floatx4 acc[CT][NB];
#pragma unroll
  for (int ct = 0; ct < CT; ++ct) {
    m_run[ct] = MINF;
    l_run[ct] = z_run[ct] = 0.f;
#pragma unroll
    for (int b = 0; b < NB; ++b) acc[ct][b] = floatx4{0.f, 0.f, 0.f, 0.f};
  }

  // edge: the tile has positions that some row of the workgroup does not attend
  auto process = [&](int t, int p, bool more, auto edge_c) __attribute__((always_inline)) {
    constexpr bool edge = decltype(edge_c)::value;
    floatx4 s[NT][CT];
#pragma unroll
    for (int k = 0; k < NT; ++k)
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) s[k][ct] = floatx4{0.f, 0.f, 0.f, 0.f};
    floatx4 sl[KHL ? NT : 1][KHL ? CT : 1];  // the low parts' products, summed apart
    if constexpr (KHL) {
#pragma unroll
      for (int k = 0; k < NT; ++k)
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) sl[k][ct] = floatx4{0.f, 0.f, 0.f, 0.f};
    }
    // All K fragments of the tile are requested at once (with hi + lo parts,
    // the registers hold one step's), and V's right after the score products,
    // so that one LDS latency is exposed per tile and V's lands during the
    // softmax.  Independent accumulators alternate between dependent products.
    half8 xk[KHL ? 1 : NS][NT];
    if constexpr (!KHL) {
#pragma unroll
      for (int d = 0; d < NS; ++d)
#pragma unroll
        for (int k = 0; k < NT; ++k) xk[d][k] = __builtin_bit_cast(half8, kb[p][(k * NS + d) * 64 + lane]);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int d = 0; d < NS; ++d) {
      if constexpr (KHL) {
        half8 xh[NT], xl[NT];
#pragma unroll
        for (int k = 0; k < NT; ++k) {
          xh[k] = __builtin_bit_cast(half8, kb[p][((k * NS + d) * KP) * 64 + lane]);
          xl[k] = __builtin_bit_cast(half8, kb[p][((k * NS + d) * KP + 1) * 64 + lane]);
        }
#pragma unroll
        for (int k = 0; k < NT; ++k)
#pragma unroll
          for (int ct = 0; ct < CT; ++ct) s[k][ct] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xh[k], qh[ct][d], s[k][ct], 0, 0, 0);
#pragma unroll
        for (int k = 0; k < NT; ++k)
#pragma unroll
          for (int ct = 0; ct < CT; ++ct) sl[k][ct] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xh[k], ql[ct][d], sl[k][ct], 0, 0, 0);
#pragma unroll
        for (int k = 0; k < NT; ++k)
#pragma unroll
          for (int ct = 0; ct < CT; ++ct) sl[k][ct] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xl[k], qh[ct][d], sl[k][ct], 0, 0, 0);
      } else {
#pragma unroll
        for (int k = 0; k < NT; ++k)
#pragma unroll
          for (int ct = 0; ct < CT; ++ct) s[k][ct] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xk[d][k], qh[ct][d], s[k][ct], 0, 0, 0);
        if constexpr (NH == 2) {
#pragma unroll
          for (int k = 0; k < NT; ++k)
#pragma unroll
            for (int ct = 0; ct < CT; ++ct) s[k][ct] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xk[d][k], ql[ct][d], s[k][ct], 0, 0, 0);
        }
      }
    }
    constexpr bool VEARLY = !VHL;
    half8 xv[VEARLY ? NP * NB : 1];
    if constexpr (VEARLY) {
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < NP * NB; ++i) xv[i] = __builtin_bit_cast(half8, vb[p][i * 64 + lane]);
      __builtin_amdgcn_sched_barrier(0);
    }
    float tf[NT][4][4];  // the tile's factors of this lane's tokens: K factor, bias, V factor, V minimum
#pragma unroll
    for (int k = 0; k < NT; ++k)
#pragma unroll
      for (int f = 0; f < 4; ++f) {
        if (!ZM && (f & 1)) continue;
        const float4 x = *reinterpret_cast<const float4*>(&tb[p][f][16 * k + 4 * g]);
        tf[k][f][0] = x.x; tf[k][f][1] = x.y; tf[k][f][2] = x.z; tf[k][f][3] = x.w;
      }
    // The next tile is requested here: behind the reads of this one, or the
    // compiler, which does not tell the two buffers apart, waits for it before
    // each of them.
    __builtin_amdgcn_sched_barrier(0);
    if (more) fetch(t + 1, p ^ 1);
    if constexpr (!KHL && NH == 1) {
      if (qlarge) {
#pragma unroll
        for (int k = 0; k < NT; ++k)
#pragma unroll
          for (int ct = 0; ct < CT; ++ct) s[k][ct] *= qs[ct];
      }
    }
    // scores: x K factor (and the column's), + bias; masked on the edges
#pragma unroll
    for (int k = 0; k < NT; ++k)
#pragma unroll
      for (int ct = 0; ct < CT; ++ct)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          float y = s[k][ct][i];
          if constexpr (KHL) y = (y + sl[k][ct][i]) * qs[ct];
          s[k][ct][i] = ZM ? __builtin_fmaf(y, tf[k][0][i], tf[k][1][i]) : y * tf[k][0][i];
        }
    if constexpr (edge) {
#pragma unroll
      for (int k = 0; k < NT; ++k)
#pragma unroll
        for (int ct = 0; ct < CT; ++ct)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int pos = t * TK + 16 * k + 4 * g + i;
            if (pos >= lim[ct] || pos < lo[ct]) s[k][ct][i] = -INFINITY;
          }
    }
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) {
      float tm = s[0][ct][0];
#pragma unroll
      for (int k = 0; k < NT; ++k)
#pragma unroll
        for (int i = 0; i < 4; ++i) tm = fmaxf(tm, s[k][ct][i]);
      tm = warp_max_q(tm);
      if (__builtin_amdgcn_ballot_w64(tm > m_run[ct] + TAU) != 0) {  // wave-uniform, rare
        const float mn = fmaxf(m_run[ct], tm);
        const float al = __builtin_amdgcn_exp2f(m_run[ct] - mn);
        m_run[ct] = mn;
        l_run[ct] *= al;
        z_run[ct] *= al;
#pragma unroll
        for (int b = 0; b < NB; ++b) acc[ct][b] *= al;
      }
    }
    // weights: p, p x V minimum kept aside, p x V factor as f16 parts
    u32x4 ph[NP][CT], pl[NH == 2 ? NP : 1][NH == 2 ? CT : 1];
#pragma unroll
    for (int k = 0; k < NT; ++k) {
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) {
        float w[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const bool hid = edge && s[k][ct][i] == -INFINITY;  // its factors may be infinite or NaN
          const float e = __builtin_amdgcn_exp2f(s[k][ct][i] - m_run[ct]);
          w[i] = e * (hid ? 0.f : tf[k][2][i]);
          s[k][ct][i] = hid ? -1.f : e;
        }
#pragma unroll
        for (int h = 0; h < 2; ++h) ph[k >> 1][ct][2 * (k & 1) + h] = pk_f16(w[2 * h], w[2 * h + 1]);
      }
    }
    // what the high parts' products leave time for: the low parts and the sums
    // (a tile's first, so that many small weights beside a large one count)
    float lt[CT], zt[CT];
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) lt[ct] = zt[ct] = 0.f;
#pragma unroll
    for (int k = 0; k < NT; ++k) {
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) {
        float r[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const bool hid = edge && s[k][ct][i] < 0.f;
          const float e = hid ? 0.f : s[k][ct][i];
          lt[ct] += e;
          if constexpr (ZM) zt[ct] = __builtin_fmaf(e, hid ? 0.f : tf[k][3][i], zt[ct]);
          const half2_t hi = __builtin_bit_cast(half2_t, (uint32_t)ph[k >> 1][ct][2 * (k & 1) + (i >> 1)]);
          if constexpr (NH == 2) r[i] = __builtin_fmaf(e, hid ? 0.f : tf[k][2][i], -(float)hi[i & 1]);
        }
        if constexpr (NH == 2) {
#pragma unroll
          for (int h = 0; h < 2; ++h) pl[k >> 1][ct][2 * (k & 1) + h] = pk_f16(r[2 * h], r[2 * h + 1]);
        }
      }
    }
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) {
      l_run[ct] += lt[ct];
      z_run[ct] += zt[ct];
    }
#pragma unroll
    for (int part = VHL ? -1 : 0; part < NH; ++part)
#pragma unroll
      for (int k = 0; k < NP; ++k)
#pragma unroll
        for (int b = 0; b < NB; ++b) {
          half8 x;
          if constexpr (VEARLY) x = xv[k * NB + b];
          else x = __builtin_bit_cast(half8, vb[p][((k * NB + b) * VP + (part < 0)) * 64 + lane]);
#pragma unroll
          for (int ct = 0; ct < CT; ++ct) {
            u32x4 pw = ph[k][ct];
            if constexpr (NH == 2) {
              if (part == 1) pw = pl[k][ct];
            }
            acc[ct][b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(x, __builtin_bit_cast(half8, pw), acc[ct][b], 0, 0, 0);
          }
        }
    // the sums are done in this block, under the matrix products
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) asm volatile("" : "+v"(l_run[ct]), "+v"(z_run[ct]));

  };

  // one barrier a tile: a buffer is refilled in the iteration after its
  // readers passed the barrier that ended theirs, and has arrived (vmcnt 0)
  // before the barrier that precedes its readers
  __builtin_amdgcn_s_waitcnt(0x0F70);
  __syncthreads();
  // tiles that some row of the workgroup attends in part, whole tiles, and again the former
  const int ta = min(max((w_from + TK - 1) / TK, tb0), tb1), tz = max(min(w_all / TK, tb1), ta);
  int p = 0, t = tb0;
  auto tiles = [&](int end, auto edge_c) __attribute__((always_inline)) {
    for (; t < end; ++t, p ^= 1) {
      process(t, p, t + 1 < tb1, edge_c);
      __builtin_amdgcn_s_waitcnt(0x0F70);
      __syncthreads();
    }
  };
#pragma unroll 1
  for (int part = 0; part < 2; ++part) {
    tiles(part == 0 ? ta : tb1, std::true_type{});
    if (part == 0) tiles(tz, std::false_type{});
  }

  // ---- output: lane (n, g) holds dims 16 b + 4 g + i of column n ----
#pragma unroll
  for (int ct = 0; ct < CT; ++ct) {
    const float L = warp_sum_q(l_run[ct]);
    const float Z = ZM ? warp_sum_q(z_run[ct]) : 0.f;
    // L == 0: no position.  A NaN score makes L NaN, which goes on to the output
    // and, with splits, through the log-sum-exp to the merge.
    const bool none = L == 0.f || (a.nan_zero != 0 && !(L > 0.f));
    const float inv = none ? 0.f : 1.f / L;
    float y[NB][4];
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int i = 0; i < 4; ++i) y[b][i] = none ? 0.f : __builtin_fmaf(acc[ct][b][i], a.vscale, Z) * inv;
    const int col = wc0 + 16 * ct + n;
    const bool live = col < ncols;
    const int r = live ? col / a.G : 0, h = kvh * a.G + (live ? col - r * a.G : 0);
    if (a.wo != nullptr) {
      const int64_t row = ((int64_t)r * a.hq + h) * a.splits_all + a.split0 + split;
      if (live) {
#pragma unroll
        for (int b = 0; b < NB; ++b)
          *reinterpret_cast<float4*>(a.wo + row * D + 16 * b + 4 * g) = make_float4(y[b][0], y[b][1], y[b][2], y[b][3]);
        if (g == 0) a.wl[row] = L == 0.f ? -INFINITY : m_run[ct] + __builtin_log2f(L);
      }
      continue;
    }
    if (a.rot != ROT_NONE) {  // H o: dim bits 0-1 and 4.. in registers, bits 2-3 across the lane rows
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        const float u0 = y[b][0] + y[b][1], u1 = y[b][0] - y[b][1], u2 = y[b][2] + y[b][3], u3 = y[b][2] - y[b][3];
        y[b][0] = u0 + u2; y[b][1] = u1 + u3; y[b][2] = u0 - u2; y[b][3] = u1 - u3;
#pragma unroll
        for (int i = 0; i < 4; ++i) y[b][i] = fwht_pair32(fwht_pair16(y[b][i], g & 1), g & 2);
      }
#pragma unroll
      for (int st = 1; st < NB; st <<= 1)
#pragma unroll
        for (int b = 0; b < NB; ++b)
          if ((b & st) == 0) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              const float u = y[b][i], v = y[b + st][i];
              y[b][i] = u + v;
              y[b + st][i] = u - v;
            }
          }
    }
    if (live) {
      const int64_t off = seq * a.o_batch + (int64_t)r * a.o_row + (int64_t)(h - seq * a.hkv_b * a.G) * a.o_head;
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        float o[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          o[i] = y[b][i] * a.oscale;
          if (a.rot == ROT_SIGNS) o[i] *= a.signs[16 * b + 4 * g + i];
        }
        if (a.ot == F32) store_small<F32, 4>(a.out, off + 16 * b + 4 * g, o);
        else if (a.ot == F16) store_small<F16, 4>(a.out, off + 16 * b + 4 * g, o);
        else store_small<BF16, 4>(a.out, off + 16 * b + 4 * g, o);
      }
    }
  }
}

// Queries of a chunk: E = D / 16 elements per lane of a 16-lane group, rotated
// (H, or x M), times qscale, to fragments of NH f16 parts.  KHL: each query is
// first scaled by the power of two that puts its largest magnitude in
// [256, 512), so that the low parts of the others stay normal f16 numbers;
// qfac takes the inverse.  NH == 1: only a query that f16 cannot hold is scaled,
// to [2^13, 2^14), and qfac is 1 for the others.
template <int D, int QT, int NH, bool KHL>
__global__ __launch_bounds__(256) void chunk_query_kernel(const void* __restrict__ query, int64_t q_batch,
                                                          int64_t q_row, int64_t q_head, int nq, int hq, int hkv, int hq_b, const float* __restrict__ signs,
                                                          const float* __restrict__ rot, int rotate, float qscale,
                                                          uint2* __restrict__ qf, int64_t qstride2,
                                                          float* __restrict__ qfac, int cstride) {
  constexpr int E = D / 16, NS = D / 32;
  __shared__ float rows[16][D + 4];
  const int grp = threadIdx.x >> 4, l16 = threadIdx.x & 15;
  const int64_t v = (int64_t)blockIdx.x * 16 + grp;
  const bool live = v < (int64_t)nq * hq;
  const int r = live ? (int)(v / hq) : 0, head = live ? (int)(v - (int64_t)r * hq) : 0;
  const int G = hq / hkv, kvh = head / G, col = r * G + head - kvh * G;
  float y[E];
  const int seq = head / hq_b;
  load_elems<QT, E>(query, seq * q_batch + (int64_t)r * q_row + (int64_t)(head - seq * hq_b) * q_head + l16 * E, y);
  if (signs != nullptr) {
#pragma unroll
    for (int i = 0; i < E; ++i) y[i] *= signs[l16 * E + i];
  }
  if (rot != nullptr) rot_matrix_lanes<D, E>(y, rot, rows[grp], l16);
  else if (rotate) fwht_lanes<E, 16>(y, l16);
  float up = 1.f;
  if constexpr (KHL || NH == 1) {
    float mx = 0.f;
#pragma unroll
    for (int i = 0; i < E; ++i) {
      y[i] *= qscale;
      mx = fmaxf(mx, fabsf(y[i]));
    }
    mx = fmaxf(mx, lane_xor<1>(mx));
    mx = fmaxf(mx, lane_xor<2>(mx));
    mx = fmaxf(mx, lane_xor<4>(mx));
    mx = fmaxf(mx, lane_xor<8>(mx));
    const int e = (int)((__float_as_uint(mx) >> 23) & 255u);  // mx in [2^(e-127), 2^(e-126))
    int ue = min(max(135 + 127 - e, 1), 253);                 // 2^(8 - (e - 127)), kept normal both ways
    if constexpr (!KHL) ue = e >= 127 + 14 && e < 255 ? 140 + 127 - e : 127;
    up = __uint_as_float((uint32_t)ue << 23);
    if (live && l16 == 0) qfac[(int64_t)kvh * cstride + col] = __uint_as_float((uint32_t)(254 - ue) << 23);
  } else {
    up = qscale;
  }
  if (!live) return;
#pragma unroll
  for (int i = 0; i < E; i += 4) {
    float x[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) x[j] = y[i + j] * up;
    const int dim = l16 * E + i, s = dim >> 5, gg = (dim >> 3) & 3, half = (dim >> 2) & 1;
    uint2* dst = qf + (int64_t)kvh * qstride2 + ((int64_t)(col >> 4) * (NS * NH * 64) + (s * NH) * 64 + gg * 16 + (col & 15)) * 2 + half;
    const uint32_t h0 = pk_f16(x[0], x[1]), h1 = pk_f16(x[2], x[3]);
    dst[0] = make_uint2(h0, h1);
    if constexpr (NH == 2)
      dst[128] = make_uint2(pk_f16(f16_rest(x[0], h0, 0), f16_rest(x[1], h0, 1)),
                            pk_f16(f16_rest(x[2], h1, 0), f16_rest(x[3], h1, 1)));
  }
}

template <int D, int NH, bool KHL>
hipError_t launch_chunk_query(const void* query, int qt, int64_t q_batch, int64_t q_row, int64_t q_head, int nq, int hq,
                              int hkv, int hq_b,
                              const float* signs, const float* rot, int rotate, float qscale, uint4* qf,
                              int64_t qstride, float* qfac, int cstride, hipStream_t st) {
  const dim3 grid((unsigned)(((int64_t)nq * hq + 15) / 16)), block(256);
  uint2* q2 = reinterpret_cast<uint2*>(qf);
  if (qt == F32) chunk_query_kernel<D, F32, NH, KHL><<<grid, block, 0, st>>>(query, q_batch, q_row, q_head, nq, hq, hkv, hq_b, signs, rot, rotate, qscale, q2, 2 * qstride, qfac, cstride);
  else if (qt == F16) chunk_query_kernel<D, F16, NH, KHL><<<grid, block, 0, st>>>(query, q_batch, q_row, q_head, nq, hq, hkv, hq_b, signs, rot, rotate, qscale, q2, 2 * qstride, qfac, cstride);
  else chunk_query_kernel<D, BF16, NH, KHL><<<grid, block, 0, st>>>(query, q_batch, q_row, q_head, nq, hq, hkv, hq_b, signs, rot, rotate, qscale, q2, 2 * qstride, qfac, cstride);
  return hipGetLastError();
}

}  // namespace ftq
