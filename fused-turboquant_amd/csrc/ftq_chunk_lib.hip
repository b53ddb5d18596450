// Attention over library-format caches (RHT with signs, Lloyd-Max codes, fp16
// norms) beyond the single-token, whole-context decode of ftq_paged.hip, on
// the kernels of ftq_chunk_kernel.h:
//   * decode steps of sliding-window layers (the last `window` positions and
//     the first `sinks`) and of head dims without a paged decode;
//   * multi-token steps: n new tokens per sequence over its compressed past
//     and over their own, unquantised, keys and values.
// The reference (hf/fused_cache.py:576-670) decodes the whole cache for these,
// expands it to the query heads and attends with torch ops.
//
// Sources: 16-token pages (ftq_paged.hip's sub-blocks) or flat rows per
// sequence ([B][Hkv][cap] codes and norms).  New keys and values are rotated
// here, scaled by a power of two per token, so that past and new tokens share
// one rotated domain and the output is un-rotated once.
//
// Two precisions.  PREC: query, K, V and weights as f16 hi + lo (~22 bits
// each) with fp32 sums -- the decode steps, whose torch form ran in float32,
// and float32 and float16 inputs.  Otherwise f16 operands with fp32 sums, for
// bfloat16 multi-token steps (whose torch form rounded the decoded cache and
// the weights to bfloat16).  float16 queries and new tokens are rounded by
// their rotation where torch took them as they are: relative error against 64
// bits 4.4e-4 with f16 operands for torch's 3.4e-4 (d = 64, 494 tokens over
// 49; queries 6 times larger 8.2e-4 for 4.1e-4), 2.1e-4 at the first precision.
#include "ftq_chunk_kernel.h"
#include "ftq_internal.h"

#include <algorithm>
#include <cmath>

namespace ftq {

float fwht_scale(int d);

namespace {

struct LibSource {
  const uint8_t* kc;        // pages, or flat K codes [B][hkv][cap][d kb / 8]
  const uint8_t* vc;        // flat V codes
  const uint16_t *kn, *vn;  // flat norms [B][hkv][cap]
  const int32_t* bt;        // pages: [B][max_blocks]
  int paged, nsub, max_blocks, cap, kb, vb;
  int64_t num_blocks;
  const int32_t* lens;      // positions of each sequence, the new tokens among them
  const float *klev, *vlev, *ksign, *vsign;
  const void *nk, *nv;      // new keys / values, or null
  int nt, n_new;            // their type and count per sequence
  int64_t k_batch, k_head, k_tok, v_batch, v_head, v_tok;
  int window, sinks, vsinks;  // decode: window (0: none), sinks, and their virtual positions (a multiple of 32)
};

// Common power of two of the weights' factors: the largest with which 2^TAU =
// 16 times the factor of the largest fp16 norm (2^16 / 2^7) stays below 2^16.
constexpr float V_LIFT = 4.f;

// bits [p, p + n) of a dword array with a pad dword, n <= 16
__device__ __forceinline__ uint32_t word_bits(const uint32_t* w, int p, int n) {
  // both words always (no branch, so that the reads of several codes overlap)
  const int i = p >> 5;
  return __builtin_amdgcn_alignbit(w[i + 1], w[i], (uint32_t)p & 31u) & ((1u << n) - 1u);
}

// One 32-token tile of one (sequence, kv head).  Virtual position v stands
// for position v, or with a window for a sink (v < vsinks) or for the
// (v - vsinks)-th position from the window's first 16-token boundary.
template <int D, bool PREC>
__global__ __launch_bounds__(256) void chunk_gather_lib_kernel(const LibSource s, int hkv, int seg0, uint4* __restrict__ kf,
                                                               int64_t kstride, uint4* __restrict__ vf, int64_t vstride,
                                                               float* __restrict__ tok, int64_t tstride) {
  constexpr int NS = D / 32, NB = D / 16, P = PREC ? 2 : 1, TK = ChunkGeo<D, PREC>::TK;
  constexpr int E = D / 16, CP = D / 8 + 1;  // codes: dwords of a row at 4 bits, one pad dword
  constexpr int VC = D / 32 + 1;             // pages: dwords of a V lane chunk at 4 bits, one pad dword
  constexpr int DP = D + 4;
  static_assert(2 * 64 * VC <= 2 * 32 * CP, "the V buffer holds either layout");
  __shared__ uint32_t krow[32][CP], vbuf[2 * 32 * CP];  // V: rows [32][CP], or lane chunks [2][64][VC]
  __shared__ __attribute__((aligned(16))) float dense[32][DP];  // new tokens' rotated K, then V
  __shared__ uint32_t tabk[16];
  __shared__ float tabv[16], inv[2], vex[32];
  __shared__ int tpos[32];  // the token's position, or -1 (hidden)
  __shared__ int tnew[32];  // its index among the new tokens, or -1
  const int tile = blockIdx.x, unit = blockIdx.y, b = unit / hkv, kvh = unit - b * hkv, tid = threadIdx.x;
  const int len = s.paged ? s.lens[b] : min(s.lens[b], s.cap), past = len - s.n_new;  // flat rows end at the capacity
  const int v0 = seg0 + tile * 32;
  const int lo = s.window > 0 ? max(0, len - s.window) : 0;
  const int kd = D * s.kb / 32, vd = D * s.vb / 32, cw = D * s.vb / 128;  // dwords: codes of a token, a V lane chunk
  const int64_t sub_bytes = 2 * D * (s.kb + s.vb) + 64;
  // position of virtual position v (negative never; it may not be attended)
  auto position = [&](int v) __attribute__((always_inline)) {
    return s.window > 0 && v >= s.vsinks ? (lo & ~15) + v - s.vsinks : v;
  };

  if (tid < 64) {
    // K table: PREC, the levels (coordinates of unit vectors) times 512 as hi +
    // lo; else the f16 values whose relative errors are closest together.  V:
    // the levels, or such f16 values.
    const int n = 1 << s.kb, m = 1 << s.vb;
    TableScale tk{512.f, 0.f}, tv{1.f, 0.f};
    if (!PREC) {
      tk = s.kb == 2 ? table_scale<4>(s.klev, true) : s.kb == 3 ? table_scale<8>(s.klev, true) : table_scale<16>(s.klev, true);
      tv = s.vb == 2 ? table_scale<4>(s.vlev, false) : s.vb == 3 ? table_scale<8>(s.vlev, false) : table_scale<16>(s.vlev, false);
    }
    if (tid < 16) {
      const float x = tk.sigma * s.klev[tid & (n - 1)], y = tv.sigma * s.vlev[tid & (m - 1)];
      const uint32_t hx = f32_to_f16_bits(x);
      tabk[tid] = hx | f32_to_f16_bits(x - f16_bits_to_f32(hx)) << 16;
      tabv[tid] = PREC ? y : f16_bits_to_f32(f32_to_f16_bits(y));
    }
    if (tid == 0) {
      inv[0] = 1.f / (tk.sigma * (1.f + tk.rmid));
      inv[1] = 1.f / (tv.sigma * (1.f + tv.rmid));
    }
  }
  // A half tile is one 16-token sub-block of a page, or 16 flat rows.
  {
    const int half = tid >> 7, u = tid & 127, hp = position(v0 + 16 * half);
    const uint8_t* base = nullptr;
    if (s.paged && hp < len) {
      const int j = hp >> 4, page = j / s.nsub;
      const int phys = page < s.max_blocks ? s.bt[(int64_t)b * s.max_blocks + page] : -1;
      if (phys >= 0 && (int64_t)phys < s.num_blocks)
        base = s.kc + (((int64_t)phys * hkv + kvh) * s.nsub + (j - page * s.nsub)) * sub_bytes;
    }
    const int64_t r0 = (int64_t)unit * s.cap + hp;
    const int rows = min(16, len - hp);  // flat rows that exist (<= 0: none)
    for (int i = u; i < 16 * kd; i += 128) {
      const int t = i / kd, w = i - t * kd;
      uint32_t x = 0;
      if (s.paged) {
        if (base != nullptr) x = reinterpret_cast<const uint32_t*>(base)[i];
      } else if (t < rows) {
        x = reinterpret_cast<const uint32_t*>(s.kc)[(r0 + t) * kd + w];
      }
      krow[16 * half + t][w] = x;
    }
    if (s.paged) {
      for (int i = u; i < 64 * cw; i += 128) {
        const int c = i / cw, w = i - c * cw;
        vbuf[(half * 64 + c) * VC + w] = base != nullptr ? reinterpret_cast<const uint32_t*>(base + 2 * D * s.kb)[i] : 0u;
      }
    } else {
      for (int i = u; i < 16 * vd; i += 128) {
        const int t = i / vd, w = i - t * vd;
        vbuf[(16 * half + t) * CP + w] = t < rows ? reinterpret_cast<const uint32_t*>(s.vc)[(r0 + t) * vd + w] : 0u;
      }
    }
    if (u < 16) {
      const int t = 16 * half + u, v = v0 + t, pos = hp + u;
      bool live = pos < len;
      if (s.window > 0) live = live && (v < s.vsinks ? pos < s.sinks && pos < lo : pos >= lo);
      const int nw = live && s.nk != nullptr && pos >= past ? pos - past : -1;
      uint32_t kn = 0, vn = 0;
      bool ok = live && nw < 0 && (!s.paged || base != nullptr);
      if (ok) {
        if (s.paged) {
          const uint16_t* nr = reinterpret_cast<const uint16_t*>(base + 2 * D * (s.kb + s.vb));
          kn = nr[u];
          vn = nr[16 + u];
        } else {
          kn = s.kn[r0 + u];
          vn = s.vn[r0 + u];
        }
      }
      tpos[t] = ok || nw >= 0 ? pos : -1;
      tnew[t] = nw;
      // V operand: level * 2^(ex + 8), near its norm; the weight's factor stays
      // near [32, 64) V_LIFT, so that small weights' low parts are normal f16
      // numbers (the 2^8 and V_LIFT leave with the accumulators' scale)
      const int ex = min(max((int)((vn >> 10) & 31u) - 20, -6), 7);
      vex[t] = __uint_as_float((uint32_t)(127 + 8 + ex) << 23);
      dense[t][0] = f16_bits_to_f32(kn);
      dense[t][1] = f16_bits_to_f32(vn) * __uint_as_float((uint32_t)(127 - ex) << 23) * V_LIFT;
    }
  }
  __syncthreads();
  float* to = tok + (int64_t)unit * tstride + (int64_t)(tile * 32 / TK) * 4 * TK + (tile * 32) % TK;
  if (tid < 32) {
    const bool ok = tpos[tid] >= 0;
    to[TK + tid] = ok ? 0.f : -INFINITY;
    to[3 * TK + tid] = 0.f;
    if (tnew[tid] < 0) {
      // an infinite norm stands for a NaN vector (its decode is infinity times the levels, rotated)
      to[tid] = ok ? dense[tid][0] * inv[0] + (dense[tid][0] - dense[tid][0]) : 0.f;
      to[2 * TK + tid] = ok ? dense[tid][1] * inv[1] : 0.f;
    }
  }
  // whether the tile holds new tokens (uniform: with new tokens v is the position)
  const bool any_new = s.nk != nullptr && v0 + 32 > past && v0 < len;
  const int l16 = tid & 15, grp = tid >> 4;
  auto rotate_new = [&](const void* src, int64_t sb, int64_t sh, int64_t st, const float* sign, bool isv) {
    for (int t = grp; t < 32; t += 16) {
      const int nw = tnew[t];
      if (nw < 0) continue;  // the 16 lanes of a group agree
      float y[E];
      const int64_t off = b * sb + kvh * sh + nw * st + l16 * E;
      if (s.nt == F32) load_elems<F32, E>(src, off, y);
      else if (s.nt == F16) load_elems<F16, E>(src, off, y);
      else load_elems<BF16, E>(src, off, y);
#pragma unroll
      for (int i = 0; i < E; ++i) y[i] *= sign[l16 * E + i];
      fwht_lanes<E, 16>(y, l16);
      float mx = 0.f, fin = 0.f;  // fin: NaN for a token with an infinity or a NaN
#pragma unroll
      for (int i = 0; i < E; ++i) {
        y[i] *= 1.f / __builtin_sqrtf((float)D);
        mx = fmaxf(mx, fabsf(y[i]));
        fin += y[i] * 0.f;
      }
      fin += lane_xor<1>(fin);
      fin += lane_xor<2>(fin);
      fin += lane_xor<4>(fin);
      fin += lane_xor<8>(fin);
      const bool ok = fin == 0.f;
      mx = fmaxf(mx, lane_xor<1>(mx));
      mx = fmaxf(mx, lane_xor<2>(mx));
      mx = fmaxf(mx, lane_xor<4>(mx));
      mx = fmaxf(mx, lane_xor<8>(mx));
      // K: largest magnitude to [512, 1024).  V: largest magnitude M to
      // [2^a, 2^(a+1)), a = log2 M + 3 within [2, 14]: the weight's factor
      // M 2^(8 - a) is then in [32, 64) V_LIFT as for the codes
      const int e = (int)((__float_as_uint(mx) >> 23) & 255u) - 127;
      const int a = isv ? min(max(e + 3, 2), 14) : 9;
      const int up = min(max(a - e + 127, 1), 253);
      const float f = __uint_as_float((uint32_t)up << 23);
#pragma unroll
      for (int i = 0; i < E; ++i) dense[t][l16 * E + i] = ok ? y[i] * f : 0.f;
      // a token that is not finite: operands of 0 and a NaN factor, so that the
      // rows that attend it are NaN and the others (whose products meet its
      // operands with a weight of 0) are not
      if (l16 == 0)
        to[(isv ? 2 * TK : 0) + t] = ok ? __uint_as_float((uint32_t)(254 - up) << 23) * (isv ? 256.f * V_LIFT : 1.f) : __builtin_nanf("");
    }
  };
  if (any_new) {
    __syncthreads();  // the norms in `dense` have been read
    rotate_new(s.nk, s.k_batch, s.k_head, s.k_tok, s.ksign, false);
    __syncthreads();
  }
  uint4* ko = kf + (int64_t)unit * kstride + (int64_t)tile * 2 * NS * P * 64;
  for (int u = tid; u < 2 * NS * 64; u += 256) {
    const int lane = u & 63, ts = u >> 6, m = lane & 15, g = lane >> 4;
    const int t = (ts / NS) * 16 + m, d0 = (ts % NS) * 32 + 8 * g;
    uint32_t h[4], l[4];
    if (any_new && tnew[t] >= 0) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float x = dense[t][d0 + 2 * j], y = dense[t][d0 + 2 * j + 1];
        h[j] = pk_f16(x, y);
        l[j] = PREC ? pk_f16(f16_rest(x, h[j], 0), f16_rest(y, h[j], 1)) : 0u;
      }
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint32_t x = tabk[word_bits(krow[t], (d0 + 2 * j) * s.kb, s.kb)];
        const uint32_t y = tabk[word_bits(krow[t], (d0 + 2 * j + 1) * s.kb, s.kb)];
        h[j] = (x & 0xffffu) | (y << 16);
        l[j] = (x >> 16) | (y & 0xffff0000u);
      }
    }
    ko[(ts * P) * 64 + lane] = make_uint4(h[0], h[1], h[2], h[3]);
    if constexpr (PREC) ko[(ts * P + 1) * 64 + lane] = make_uint4(l[0], l[1], l[2], l[3]);
  }
  if (any_new) {
    __syncthreads();
    rotate_new(s.nv, s.v_batch, s.v_head, s.v_tok, s.vsign, true);
    __syncthreads();
  }
  uint4* vo = vf + (int64_t)unit * vstride + (int64_t)tile * NB * P * 64;
  for (int u = tid; u < NB * 64; u += 256) {
    const int lane = u & 63, bb = u >> 6, m = lane & 15, g = lane >> 4, d = 16 * bb + m;
    uint32_t h[4], l[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      float x[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int ti = 2 * (j & 1) + i, t = (j >> 1) * 16 + 4 * g + ti;
        if (any_new && tnew[t] >= 0) {
          x[i] = dense[t][d];
        } else {
          const uint32_t c = s.paged ? word_bits(vbuf + ((j >> 1) * 64 + lane) * VC, (4 * bb + ti) * s.vb, s.vb)
                                     : word_bits(vbuf + t * CP, d * s.vb, s.vb);
          x[i] = tabv[c] * vex[t];
        }
      }
      h[j] = pk_f16(x[0], x[1]);
      l[j] = PREC ? pk_f16(f16_rest(x[0], h[j], 0), f16_rest(x[1], h[j], 1)) : 0u;
    }
    vo[(bb * P) * 64 + lane] = make_uint4(h[0], h[1], h[2], h[3]);
    if constexpr (PREC) vo[(bb * P + 1) * 64 + lane] = make_uint4(l[0], l[1], l[2], l[3]);
  }
}

struct LibPlan {
  int cols, tk, seg, nseg, splits, vsinks, span;
  int64_t colpad, kstride, vstride, tstride, qstride;
  int64_t o_k, o_v, o_t, o_q, o_f, o_o, o_l, bytes;
};

constexpr int64_t kLibSegBytes = (int64_t)192 << 20;

// max_len: longest sequence, the new tokens among them
bool lib_plan(LibPlan& p, int batch, int nq, int hq, int hkv, int d, int max_len, int window, int sinks, bool prec,
              bool decode) {
  if (batch <= 0 || nq <= 0 || hq <= 0 || hkv <= 0 || hq % hkv != 0 || hq / hkv > 16 || max_len < 0 || max_len > (1 << 30) ||
      window < 0 || sinks < 0)
    return false;
  const int64_t units = (int64_t)batch * hkv, ncols = (int64_t)nq * (hq / hkv);
  if (units > 65535 || ncols > ((int64_t)1 << 30)) return false;
  p.cols = d == 256 ? 64 : 128;
  p.tk = d == 64 ? 64 : 32;
  p.colpad = (ncols + p.cols - 1) / p.cols * p.cols;
  p.vsinks = 0;
  int64_t span = max_len;
  if (decode && window > 0) {
    // virtual positions: the sinks, then the window from its 16-token boundary
    p.vsinks = (int)(((int64_t)std::min(sinks, max_len) + 31) / 32 * 32);
    span = p.vsinks + std::min<int64_t>(max_len, (int64_t)window + 15);
  }
  span = std::max<int64_t>((span + 63) / 64 * 64, 64);
  if (span > (1 << 30)) return false;
  p.span = (int)span;
  const int parts_kv = prec ? 4 : 2;
  const int64_t per_token = units * (d * 2 * parts_kv + 16);
  int64_t seg = std::max<int64_t>(kLibSegBytes / per_token / 64 * 64, 1024);
  if (seg > span) seg = span;
  p.seg = (int)seg;
  p.nseg = (int)((span + seg - 1) / seg);
  const int64_t wgs = units * (p.colpad / p.cols);
  int64_t s = std::min<int64_t>(512 / wgs, seg / p.tk / 4);
  p.splits = (int)std::min<int64_t>(std::max<int64_t>(s, 1), 32);
  const int64_t t16 = p.seg / 16;
  p.kstride = t16 * (d / 32) * (prec ? 2 : 1) * 64;
  p.vstride = t16 / 2 * (d / 16) * (prec ? 2 : 1) * 64;
  p.tstride = (int64_t)p.seg * 4;
  p.qstride = p.colpad / 16 * (d / 32) * (prec ? 2 : 1) * 64;
  int64_t at = 0;
  auto take = [&](int64_t bytes) {
    const int64_t o = at;
    at += (bytes + 255) / 256 * 256;
    return o;
  };
  p.o_k = take(p.kstride * units * 16);
  p.o_v = take(p.vstride * units * 16);
  p.o_t = take(p.tstride * units * 4);
  p.o_q = take(p.qstride * units * 16);
  p.o_f = take(p.colpad * units * 4);
  const int64_t all = (int64_t)p.nseg * p.splits, rows = (int64_t)nq * hq * batch * all;
  p.o_o = take(all > 1 ? rows * d * 4 : 0);
  p.o_l = take(all > 1 ? rows * 4 : 0);
  p.bytes = at;
  return true;
}

// Splits (and segments) of the rows meet here and leave for their strided
// places; the un-rotation is the merge's.  One wave per row.
template <int D, int OT>
__global__ __launch_bounds__(256) void chunk_merge_kernel(const float* __restrict__ wo, const float* __restrict__ wl,
                                                          int64_t rows, int hq_all, int hq_b, int splits,
                                                          const float* __restrict__ signs, float scale,
                                                          void* __restrict__ out, int64_t o_batch, int64_t o_row,
                                                          int64_t o_head, int nan_zero) {
  constexpr int E = D / 64;
  const int lane = threadIdx.x & 63;
  const int64_t r = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (r >= rows) return;
  const float* lse = wl + r * splits;
  const float* po = wo + r * splits * D + lane * E;
  float M = -INFINITY;
  bool nan = false;  // a split with a NaN score; the maximum does not show it
  for (int s = lane; s < splits; s += 64) {
    M = fmaxf(M, lse[s]);
    nan = nan || lse[s] != lse[s];
  }
  M = wave_max64(M);
  nan = __builtin_amdgcn_ballot_w64(nan) != 0;
  float y[E], W = 0.f;
#pragma unroll
  for (int i = 0; i < E; ++i) y[i] = 0.f;
  if (nan) {
#pragma unroll
    for (int i = 0; i < E; ++i) y[i] = nan_zero ? 0.f : __builtin_nanf("");
    W = 1.f;
  } else if (M != -INFINITY) {
    for (int s = 0; s < splits; ++s) {
      float x[E];
      load_f32_small<E>(po + (int64_t)s * D, x);
      const float w = __builtin_amdgcn_exp2f(lse[s] - M);
      W += w;
#pragma unroll
      for (int i = 0; i < E; ++i) y[i] = __builtin_fmaf(w, x[i], y[i]);
    }
  }
  const float inv = W > 0.f ? 1.f / W : 0.f;
#pragma unroll
  for (int i = 0; i < E; ++i) y[i] *= inv;
  fwht_wave64<E>(y, lane);
#pragma unroll
  for (int i = 0; i < E; ++i) y[i] = y[i] * scale * signs[lane * E + i];
  const int64_t row = r / hq_all;
  const int h = (int)(r - row * hq_all), b = h / hq_b;
  store_small<OT, E>(out, b * o_batch + row * o_row + (int64_t)(h - b * hq_b) * o_head + lane * E, y);
}

template <int D, bool PREC>
hipError_t lib_launch(const LibPlan& p, LibSource s, const void* q, int qt, int64_t q_batch, int64_t q_row, int64_t q_head,
                      int batch, int nq, int hq, int hkv, int max_len, float scale, uint8_t* ws, void* out, int ot,
                      int64_t o_batch, int64_t o_row, int64_t o_head, hipStream_t st) {
  constexpr int NH = PREC ? 2 : 1;
  const bool decode = s.nk == nullptr;
  uint4* kf = reinterpret_cast<uint4*>(ws + p.o_k);
  uint4* vf = reinterpret_cast<uint4*>(ws + p.o_v);
  uint4* qf = reinterpret_cast<uint4*>(ws + p.o_q);
  float* tok = reinterpret_cast<float*>(ws + p.o_t);
  float* qfac = reinterpret_cast<float*>(ws + p.o_f);
  const int units = batch * hkv;
  const float rs = fwht_scale(D);
  hipError_t e = launch_chunk_query<D, NH, PREC>(q, qt, q_batch, q_row, q_head, nq, batch * hq, units, hq, s.ksign, nullptr, 1,
                                                 rs * scale * 1.4426950408889634f, qf, p.qstride, qfac, (int)p.colpad, st);
  if (e != hipSuccess) return e;
  ChunkAttn a{};
  a.kf = reinterpret_cast<const u32x4*>(kf);
  a.vf = reinterpret_cast<const u32x4*>(vf);
  a.qf = reinterpret_cast<const u32x4*>(qf);
  a.tok = tok; a.qfac = qfac;
  a.kstride = p.kstride; a.vstride = p.vstride; a.qstride = p.qstride; a.tstride = p.tstride; a.cstride = (int)p.colpad;
  a.nq = nq; a.G = hq / hkv; a.hq = batch * hq; a.hkv = units; a.hkv_b = hkv;
  a.splits = p.splits; a.splits_all = p.splits * p.nseg;
  s.vsinks = p.vsinks;
  if (decode && s.window > 0) {  // virtual positions, hidden ones by their bias
    a.lens = nullptr; a.past = p.span - 1; a.window = 0;
  } else {
    a.lens = s.lens; a.lens_less = nq; a.past = max_len - nq; a.window = decode ? 0 : s.window;
  }
  if (!decode) s.window = 0;  // virtual positions are a decode step's
  a.vscale = 1.f / (256.f * V_LIFT);
  const bool direct = a.splits_all == 1;
  a.wo = direct ? nullptr : reinterpret_cast<float*>(ws + p.o_o);
  a.wl = direct ? nullptr : reinterpret_cast<float*>(ws + p.o_l);
  a.out = out; a.ot = ot; a.rot = ROT_SIGNS; a.signs = s.vsign; a.oscale = rs;
  a.o_batch = o_batch; a.o_row = o_row; a.o_head = o_head;
  a.nan_zero = decode;
  for (int i = 0; i < p.nseg; ++i) {
    a.seg0 = i * p.seg;
    a.seg1 = std::min(a.seg0 + p.seg, p.span);
    a.split0 = i * p.splits;
    chunk_gather_lib_kernel<D, PREC><<<dim3((a.seg1 - a.seg0) / 32, units), dim3(256), 0, st>>>(
        s, hkv, a.seg0, kf, p.kstride, vf, p.vstride, tok, p.tstride);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    // A decode step hides positions by their bias (ZM); a multi-token step's
    // f16 form has none to hide below its causal limits and skips the bias.
    const dim3 agrid((unsigned)(units * (p.colpad / p.cols)), p.splits);
    if (decode || PREC) chunk_attn_kernel<D, NH, PREC, PREC, true><<<agrid, dim3(256), 0, st>>>(a);
    else chunk_attn_kernel<D, NH, PREC, PREC, PREC><<<agrid, dim3(256), 0, st>>>(a);
    if ((e = hipGetLastError()) != hipSuccess) return e;
  }
  if (direct) return hipSuccess;
  const int64_t rows = (int64_t)nq * batch * hq;
  const dim3 grid((unsigned)((rows + 3) / 4)), block(256);
  if (ot == F32) chunk_merge_kernel<D, F32><<<grid, block, 0, st>>>(a.wo, a.wl, rows, batch * hq, hq, a.splits_all, s.vsign, rs, out, o_batch, o_row, o_head, a.nan_zero);
  else if (ot == F16) chunk_merge_kernel<D, F16><<<grid, block, 0, st>>>(a.wo, a.wl, rows, batch * hq, hq, a.splits_all, s.vsign, rs, out, o_batch, o_row, o_head, a.nan_zero);
  else chunk_merge_kernel<D, BF16><<<grid, block, 0, st>>>(a.wo, a.wl, rows, batch * hq, hq, a.splits_all, s.vsign, rs, out, o_batch, o_row, o_head, a.nan_zero);
  return hipGetLastError();
}

}  // namespace
}  // namespace ftq

using namespace ftq;

extern "C" int64_t ftq_lib_attention_workspace_bytes(int batch, int n_query, int num_q_heads, int num_kv_heads, int d,
                                                     int max_len, int window, int sinks, int precise, int decode) {
  LibPlan p;
  if (!(d == 64 || d == 128 || d == 256) ||
      !lib_plan(p, batch, n_query, num_q_heads, num_kv_heads, d, max_len, window, sinks, precise != 0, decode != 0))
    return -1;
  return p.bytes;
}

extern "C" int ftq_lib_attention(const ftq_lib_attention_args* x, void* workspace, int64_t workspace_bytes, void* stream) {
  FTQ_REQUIRE(x != nullptr, "null pointer argument");
  const int d = x->d;
  FTQ_REQUIRE(d == 64 || d == 128 || d == 256, "library attention: head_dim must be 64, 128 or 256");
  FTQ_REQUIRE(x->bits_k >= 2 && x->bits_k <= 4 && x->bits_v >= 2 && x->bits_v <= 4, "bits must be 2, 3, or 4");
  FTQ_REQUIRE(x->batch >= 0 && x->n_query >= 0 && x->max_len >= x->n_query, "bad batch / token counts");
  if (x->batch == 0 || x->n_query == 0) return FTQ_OK;
  const bool decode = x->new_key == nullptr;
  FTQ_REQUIRE(decode ? x->n_query == 1 : x->new_value != nullptr, "one query token without new keys; new keys come with new values");
  FTQ_REQUIRE(!(x->paged && d == 64), "pages hold head_dim 128 or 256");
  FTQ_REQUIRE(!x->paged || (x->page_size >= 16 && x->page_size % 16 == 0), "page_size must be a multiple of 16");
  FTQ_REQUIRE(x->max_blocks >= 0 && x->num_blocks >= 0 && x->capacity >= 0, "bad block counts");
  FTQ_REQUIRE(x->paged || x->capacity >= x->max_len, "capacity is smaller than max_len");
  FTQ_REQUIRE(x->query && x->out && x->lens && x->k_signs && x->v_signs && x->k_levels && x->v_levels && x->codes_k && workspace,
              "null pointer argument");
  FTQ_REQUIRE(x->paged ? x->block_table != nullptr : (x->codes_v && x->norms_k && x->norms_v), "null pointer argument");
  FTQ_REQUIRE(x->q_dtype >= F32 && x->q_dtype <= BF16 && x->out_dtype >= F32 && x->out_dtype <= BF16 &&
                  (decode || (x->new_dtype >= F32 && x->new_dtype <= BF16)),
              "dtype must be FTQ_F32, FTQ_F16 or FTQ_BF16");
  FTQ_REQUIRE(aligned16(x->query) && aligned16(x->out) && aligned16(workspace) && aligned4(x->codes_k) && aligned4(x->codes_v) &&
                  (decode || (aligned16(x->new_key) && aligned16(x->new_value))),
              "query, out, new keys / values and workspace must be 16-byte aligned, codes 4-byte aligned");
  // 16-byte (or, 4 elements of a 16-bit type, 8-byte) accesses along every stride
  const int64_t strides = x->q_batch | x->q_row | x->q_head | x->o_batch | x->o_row | x->o_head |
                          (decode ? 0 : x->k_batch | x->k_head | x->k_tok | x->v_batch | x->v_head | x->v_tok);
  FTQ_REQUIRE((strides & 7) == 0, "strides must be multiples of 8 elements");
  LibPlan p;
  const bool prec = x->precise != 0;
  FTQ_REQUIRE(lib_plan(p, x->batch, x->n_query, x->num_q_heads, x->num_kv_heads, d, x->max_len, x->window, x->sinks, prec, decode),
              "library attention: bad head counts or too many tokens");
  FTQ_REQUIRE(workspace_bytes >= p.bytes, "workspace too small (see ftq_lib_attention_workspace_bytes)");
  LibSource s{};
  s.kc = x->codes_k; s.vc = x->codes_v; s.kn = x->norms_k; s.vn = x->norms_v; s.bt = x->block_table;
  s.paged = x->paged != 0; s.nsub = x->paged ? x->page_size / 16 : 1; s.max_blocks = x->max_blocks; s.cap = x->capacity;
  s.kb = x->bits_k; s.vb = x->bits_v; s.num_blocks = x->num_blocks; s.lens = x->lens;
  s.klev = x->k_levels; s.vlev = x->v_levels; s.ksign = x->k_signs; s.vsign = x->v_signs;
  s.nk = x->new_key; s.nv = x->new_value; s.nt = x->new_dtype; s.n_new = decode ? 0 : x->n_query;
  s.k_batch = x->k_batch; s.k_head = x->k_head; s.k_tok = x->k_tok;
  s.v_batch = x->v_batch; s.v_head = x->v_head; s.v_tok = x->v_tok;
  s.window = x->window; s.sinks = x->sinks;
  if (!decode) s.sinks = 0;
  uint8_t* ws = static_cast<uint8_t*>(workspace);
  hipStream_t st = (hipStream_t)stream;
#define FTQ_LIB_GO(D, PR)                                                                                              \
  lib_launch<D, PR>(p, s, x->query, x->q_dtype, x->q_batch, x->q_row, x->q_head, x->batch, x->n_query, x->num_q_heads, \
                    x->num_kv_heads, x->max_len, x->scale, ws, x->out, x->out_dtype, x->o_batch, x->o_row, x->o_head, st)
  hipError_t e;
  if (prec) e = d == 64 ? FTQ_LIB_GO(64, true) : d == 128 ? FTQ_LIB_GO(128, true) : FTQ_LIB_GO(256, true);
  else e = d == 64 ? FTQ_LIB_GO(64, false) : d == 128 ? FTQ_LIB_GO(128, false) : FTQ_LIB_GO(256, false);
#undef FTQ_LIB_GO
  return hip_status(e);
}
