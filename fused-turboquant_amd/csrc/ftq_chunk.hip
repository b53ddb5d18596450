// Chunk attention over the vLLM v1 slot cache and the raw fp16 slots of the
// boundary layers: n consecutive query tokens of one sequence, whose K and V
// are already in their slots, attend the stored positions (the reference's
// continuation prefill, vllm_plugin/v1_backend.py:1359-1384, which runs its
// decode kernel over one synthetic sequence per query token).  Kernels and
// fragment layout: ftq_chunk_kernel.h.
#include "ftq_chunk_kernel.h"
#include "ftq_internal.h"
#include "ftq_v1_dev.h"

#include <algorithm>
#include <cmath>

namespace ftq {

float fwht_scale(int d);
bool v1_widths_ok(int kb, int vb, int flags);

namespace {

constexpr int KB_RAW = 16;  // key_bits of raw fp16 slots

// n <= 16 bits at bit offset p of a little-endian dword row (one pad dword)
__device__ __forceinline__ uint32_t row_bits(const uint32_t* row, int p, int n) {
  // both words always (no branch, so that the reads of several codes overlap)
  const int i = p >> 5;
  return __builtin_amdgcn_alignbit(row[i + 1], row[i], (uint32_t)p & 31u) & ((1u << n) - 1u);
}

__device__ __forceinline__ float e4m3_value(uint32_t b) {
  const uint32_t e = (b >> 3) & 15u, m = b & 7u;
  float v;
  if (e == 0) v = (float)m * (1.f / 512.f);
  else if (e == 15 && m == 7) v = __builtin_nanf("");
  else v = __uint_as_float(((e + 120u) << 23) | (m << 20));
  return (b & 0x80u) ? -v : v;
}

// power of two that puts the largest |c| of n table entries in [512, 1024)
__device__ __forceinline__ float table_pow2(const float* __restrict__ c, int n) {
  float mx = 0.f;
  for (int i = (int)(threadIdx.x & 63u); i < n; i += 64) mx = fmaxf(mx, fabsf(c[i]));
  mx = wave_max64(mx);
  if (!(mx > 0.f) || !(mx < INFINITY)) return 1.f;
  const int e = (int)((__float_as_uint(mx) >> 23) & 255u);
  return __uint_as_float((uint32_t)min(max(263 - e, 1), 254) << 23);
}

// Common power of two of the weights' factors (the V scale's own power of two
// is in the V operand, so that a factor is in [1, 2) times this; raw slots have
// no scale): the largest with which 2^TAU = 16 times a factor stays an f16
// number, so that the weights' low parts are normal numbers as far down as f16
// has them.  With the tile-first sums of the attention kernel, one key that
// takes most of the weight over 30000 others 24 log2 units below it, relative
// error of raw d = 64 / K4 V4 d = 64 / K8 V8 d = 256 with factors of 1 / 32 /
// 32 and one running sum: 1.8e-5 / 1.2e-5 / 1.3e-5; now 1.0e-6 / 8e-7 / 8e-7.
__host__ __device__ constexpr float v_lift(bool raw, int vb) { return raw ? 2048.f : vb == 8 ? 512.f : 1024.f; }

// One 32-token tile of one kv head: slots -> LDS rows -> fragments.
template <int D, bool KHL>
__global__ __launch_bounds__(256) void chunk_gather_v1_kernel(
    const uint8_t* __restrict__ cache, int64_t num_blocks, int lbs, int64_t s_blk, int64_t s_pos, int64_t s_head,
    const int32_t* __restrict__ bt_row, int max_blocks, const float* __restrict__ cent, int kb, int vb, int kf8,
    int seg0, int total, int pitch, int wide, uint4* __restrict__ kf, int64_t kstride, uint4* __restrict__ vf, int64_t vstride,
    float* __restrict__ tok, int64_t tstride) {
  constexpr int NS = D / 32, NB = D / 16, KP = KHL ? 2 : 1, TK = ChunkGeo<D, KHL>::TK;
  extern __shared__ __attribute__((aligned(16))) uint32_t rows[];  // [32][pitch]
  __shared__ uint32_t tab[256];   // f16 hi | lo << 16 of the scaled table values
  __shared__ float tabn[256];     // the value the K norm correction sums the squares of
  __shared__ int tok_ok[32];
  __shared__ float vex[32];       // 2^e of the token's V operand
  __shared__ float tab_scale_inv;
  const int tile = blockIdx.x, kvh = blockIdx.y, tid = threadIdx.x;
  const bool raw = kb == KB_RAW;
  const V1Geom geo = raw ? V1Geom{2 * D, 2 * D, 2 * D, 4 * D} : v1_geom(D, kb, vb, kf8 != 0);
  const int nd = (geo.raw + 3) / 4;
  const float mid = raw ? 0.f : 0.5f * (float)((1 << vb) - 1);
  const int pos0 = seg0 + tile * 32;

  float beyond = 0.f;  // raw slots: whether this lane read a V element that is not finite
  {  // 8 lanes a token, 16 bytes (or 4 dwords) each
    const int t = tid >> 3, sub = tid & 7;
    const int pos = pos0 + t, page = pos >> lbs;
    const int phys = (pos < total && page < max_blocks) ? bt_row[page] : -1;
    const bool ok = phys >= 0 && (int64_t)phys < num_blocks;
    const int64_t off = ok ? (int64_t)phys * s_blk + (int64_t)(pos & ((1 << lbs) - 1)) * s_pos + (int64_t)kvh * s_head : 0;
    const uint32_t* src = reinterpret_cast<const uint32_t*>(cache + off);
    uint32_t* dst = rows + t * pitch;
    for (int c = sub; c * 4 < nd; c += 8) {
      uint32_t w[4] = {0u, 0u, 0u, 0u};
      if (ok) {
        if (wide && 16 * (c + 1) <= s_head) {  // inside the slot's stride
          const uint4 x = *reinterpret_cast<const uint4*>(src + 4 * c);
          w[0] = x.x; w[1] = x.y; w[2] = x.z; w[3] = x.w;
        } else {
#pragma unroll
          for (int j = 0; j < 4; ++j) w[j] = 4 * c + j < nd ? src[4 * c + j] : 0u;
        }
      }
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (4 * c + j < nd) dst[4 * c + j] = w[j];
      if (raw && c >= D / 8) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if ((w[j] & 0x7c00u) == 0x7c00u || (w[j] & 0x7c000000u) == 0x7c000000u) beyond = 1.f;
      }
    }
    if (sub == 0) tok_ok[t] = ok;
  }
  if (!raw && tid < 64) {
    float sg = 1.f;
    if (kf8) sg = 1.f;
    else if (KHL) sg = table_pow2(cent, 1 << kb);
    else if (kb == 2) sg = table_scale<4>(cent, true).sigma;
    else if (kb == 3) sg = table_scale<8>(cent, true).sigma;
    else sg = table_scale<16>(cent, true).sigma;
    for (int e = tid; e < (1 << kb); e += 64) {
      const float c = kf8 ? e4m3_value((uint32_t)e) : cent[e], x = sg * c;
      const uint32_t h = f32_to_f16_bits(x);
      const float hv = f16_bits_to_f32(h);
      tab[e] = h | (KHL ? f32_to_f16_bits(x - hv) << 16 : 0u);
      tabn[e] = KHL ? c : hv;
    }
    if (tid == 0) tab_scale_inv = KHL ? 1.f / sg : 1.f;
  }
  __syncthreads();

  {  // per-token factors: 8 lanes a token share the K norm's sum
    const int t = tid >> 3, sub = tid & 7;
    const uint32_t* row = rows + t * pitch;
    float csq = 0.f;
    if (!raw && !kf8) {
#pragma unroll 8
      for (int d = 0; d < D / 8; ++d) {
        const float c = tabn[row_bits(row, (sub * (D / 8) + d) * kb, kb)];
        csq = __builtin_fmaf(c, c, csq);
      }
      csq = group_sum<8>(csq);
    }
    if (raw) beyond = group_sum<8>(beyond);
    if (sub == 0) {
      const bool ok = tok_ok[t] != 0;
      // A raw V that is not finite (a bf16 value beyond fp16's range): operands of
      // 0 and a NaN factor, so that the rows that attend it are NaN and those
      // whose products only meet it with a weight of 0 are not.
      float fk = 1.f, vs = beyond == 0.f ? v_lift(true, vb) : __builtin_nanf(""), vm = 0.f, ve = beyond == 0.f ? 1.f : 0.f;
      if (!raw) {
        if (!kf8) {
          const float kn = f16_bits_to_f32(row_bits(row, 8 * geo.mse, 16));
          fk = KHL ? kn / __builtin_sqrtf(csq + 1e-16f) * tab_scale_inv : kn * __builtin_amdgcn_rsqf(csq + 1e-16f);
        }
        const uint32_t sb = row_bits(row, 8 * (geo.kps + geo.vdb), 16);
        // V operand (code - mid) * 2^e, exact in f16, with the middle of the
        // code range moved into the minimum: the sums then have the outputs'
        // magnitude, not that of an offset the minimum cancels.  2^(e + 5) is the scale's own power
        // of two, and e is held where the largest code stays finite and the
        // codes normal
        const int e = min(max((int)((sb >> 10) & 31u) - 20, -14), vb == 8 ? 9 : 12);
        ve = __uint_as_float((uint32_t)(127 + e) << 23);
        vs = f16_bits_to_f32(sb) * __uint_as_float((uint32_t)(127 - e) << 23) * (v_lift(false, vb) / 32.f);
        vm = __builtin_fmaf(mid, f16_bits_to_f32(sb), f16_bits_to_f32(row_bits(row, 8 * (geo.kps + geo.vdb) + 16, 16)));
      }
      float* o = tok + (int64_t)kvh * tstride + (int64_t)(tile * 32 / TK) * 4 * TK + (tile * 32) % TK + t;
      o[0] = ok ? fk : 0.f;
      o[TK] = ok ? 0.f : -INFINITY;
      o[2 * TK] = ok ? vs : 0.f;
      o[3 * TK] = ok ? vm : 0.f;
      vex[t] = ve;
    }
  }
  __syncthreads();

  // K fragments: unit u = (16-token tile, step, lane)
  uint4* ko = kf + (int64_t)kvh * kstride + (int64_t)tile * 2 * NS * KP * 64;
  for (int u = tid; u < 2 * NS * 64; u += 256) {
    const int lane = u & 63, ts = u >> 6, m = lane & 15, g = lane >> 4;
    const int t = (ts / NS) * 16 + m, d0 = (ts % NS) * 32 + 8 * g;
    const uint32_t* row = rows + t * pitch;
    uint32_t h[4], l[4];
    if (raw) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        h[j] = row[d0 / 2 + j];
        l[j] = 0;
      }
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint32_t a = tab[row_bits(row, (d0 + 2 * j) * kb, kb)], b = tab[row_bits(row, (d0 + 2 * j + 1) * kb, kb)];
        h[j] = (a & 0xffffu) | (b << 16);
        l[j] = (a >> 16) | (b & 0xffff0000u);
      }
    }
    ko[(ts * KP) * 64 + lane] = make_uint4(h[0], h[1], h[2], h[3]);
    if constexpr (KHL) ko[(ts * KP + 1) * 64 + lane] = make_uint4(l[0], l[1], l[2], l[3]);
  }
  // V fragments: unit u = (16-dim block, lane)
  uint4* vo = vf + (int64_t)kvh * vstride + (int64_t)tile * NB * 64;
  for (int u = tid; u < NB * 64; u += 256) {
    const int lane = u & 63, b = u >> 6, m = lane & 15, g = lane >> 4, d = 16 * b + m;
    uint32_t w[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int t = (j >> 1) * 16 + 4 * g + 2 * (j & 1);
      if (raw) {
        w[j] = (vex[t] != 0.f ? row_bits(rows + t * pitch, 16 * D + 16 * d, 16) : 0u) |
               (vex[t + 1] != 0.f ? row_bits(rows + (t + 1) * pitch, 16 * D + 16 * d, 16) << 16 : 0u);
      } else {
        const float x = ((float)row_bits(rows + t * pitch, 8 * geo.kps + d * vb, vb) - mid) * vex[t];
        const float y = ((float)row_bits(rows + (t + 1) * pitch, 8 * geo.kps + d * vb, vb) - mid) * vex[t + 1];
        w[j] = pk_f16(x, y);
      }
    }
    vo[b * 64 + lane] = make_uint4(w[0], w[1], w[2], w[3]);
  }
}

// What a call of n_query tokens over positions [0, past + n_query) needs.
struct ChunkPlan {
  int khl, cols, tk, base, seg, nseg, splits;  // base: first token read; seg: tokens per segment
  int64_t colpad, kstride, vstride, tstride, qstride;
  int64_t o_k, o_v, o_t, o_q, o_f, o_o, o_l, bytes;  // offsets into the workspace
};

constexpr int64_t kSegBytes = (int64_t)192 << 20;  // dequantised fragments held at once

// false: a count is out of range.  need_ws: the output goes through the merge
// even with one split (a caller's rotation matrix).
bool chunk_plan(ChunkPlan& p, int nq, int hq, int hkv, int d, int past, int kb, int vb, int flags, int window,
                bool need_ws) {
  if (nq <= 0 || hq <= 0 || hkv <= 0 || hq % hkv != 0 || past < 0 || (int64_t)past + nq > (1 << 30)) return false;
  const bool raw = kb == KB_RAW;
  p.khl = !(d == 128 && (raw || ((flags & V1F_KFP8) == 0 && kb >= 2 && kb <= 4 && vb >= 2 && vb <= 4)));
  p.cols = d == 256 ? 64 : 128;
  p.tk = d == 64 ? 64 : 32;
  const int64_t ncols = (int64_t)nq * (hq / hkv);
  if (ncols > ((int64_t)1 << 30)) return false;
  p.colpad = (ncols + p.cols - 1) / p.cols * p.cols;
  p.base = window > 0 ? std::max(0, past + 1 - window) / 64 * 64 : 0;
  const int total = past + nq;
  const int64_t per_token = (int64_t)hkv * (d * 2 * (p.khl ? 3 : 2) + 16);
  int64_t seg = std::max<int64_t>(kSegBytes / per_token / 64 * 64, 1024);
  const int span = (total - p.base + 63) / 64 * 64;
  if (seg > span) seg = span;
  p.seg = (int)seg;
  p.nseg = (int)((span + seg - 1) / seg);
  // splits: 512 workgroups, two per CU, and at least 4 tiles each.  At d = 256
  // LDS holds one per CU: two rounds (256 tokens over 5120, 8 heads over 4, 73 us;
  // 65 with 256 workgroups; 64 tokens 43 and 44).
  const int64_t wgs = (int64_t)hkv * (p.colpad / p.cols);
  int64_t s = 512 / wgs;
  s = std::min<int64_t>(s, p.seg / p.tk / 4);
  p.splits = (int)std::min<int64_t>(std::max<int64_t>(s, 1), 32);
  const int64_t t16 = p.seg / 16;
  p.kstride = t16 * (d / 32) * (p.khl ? 2 : 1) * 64;
  p.vstride = t16 / 2 * (d / 16) * 64;
  p.tstride = (int64_t)p.seg * 4;
  p.qstride = p.colpad / 16 * (d / 32) * 2 * 64;
  const bool parts = need_ws || p.nseg * p.splits > 1;
  int64_t at = 0;
  auto take = [&](int64_t bytes) {
    const int64_t o = at;
    at += (bytes + 255) / 256 * 256;
    return o;
  };
  p.o_k = take(p.kstride * hkv * 16);
  p.o_v = take(p.vstride * hkv * 16);
  p.o_t = take(p.tstride * hkv * 4);
  p.o_q = take(p.qstride * hkv * 16);
  p.o_f = take(p.khl ? p.colpad * hkv * 4 : 0);
  const int64_t rows = (int64_t)nq * hq * p.nseg * p.splits;
  p.o_o = take(parts ? rows * d * 4 : 0);
  p.o_l = take(parts ? rows * 4 : 0);
  p.bytes = at;
  return true;
}

template <int D, bool KHL>
hipError_t chunk_launch(const ChunkPlan& p, const void* q, int qt, int64_t q_row, int64_t q_head, const uint8_t* cache,
                        int64_t nb, int lbs, int64_t sblk, int64_t spos, int64_t shead, const int32_t* bt, int mb,
                        int past, int nq, int hq, int hkv, const float* cent, int kb, int vb, int flags, float scale,
                        int window, uint8_t* ws, void* out, int ot, int64_t o_row, int64_t o_head, const float* rot,
                        hipStream_t st) {
  const bool raw = kb == KB_RAW, vrot = (flags & V1F_VROT) != 0;
  ChunkAttn a{};
  uint4* kf = reinterpret_cast<uint4*>(ws + p.o_k);
  uint4* vf = reinterpret_cast<uint4*>(ws + p.o_v);
  uint4* qf = reinterpret_cast<uint4*>(ws + p.o_q);
  float* tok = reinterpret_cast<float*>(ws + p.o_t);
  float* qfac = reinterpret_cast<float*>(ws + p.o_f);
  const int total = past + nq;
  const float qscale = (raw || rot != nullptr ? 1.f : fwht_scale(D)) * scale * 1.4426950408889634f;
  hipError_t e = launch_chunk_query<D, 2, KHL>(q, qt, 0, q_row, q_head, nq, hq, hkv, hq, nullptr, rot, raw ? 0 : 1, qscale, qf,
                                               p.qstride, qfac, (int)p.colpad, st);
  if (e != hipSuccess) return e;
  a.kf = reinterpret_cast<const u32x4*>(kf);
  a.vf = reinterpret_cast<const u32x4*>(vf);
  a.qf = reinterpret_cast<const u32x4*>(qf);
  a.tok = tok; a.qfac = qfac;
  a.kstride = p.kstride; a.vstride = p.vstride; a.qstride = p.qstride; a.tstride = p.tstride; a.cstride = (int)p.colpad;
  a.nq = nq; a.G = hq / hkv; a.hq = hq; a.hkv = hkv; a.past = past; a.window = window;
  a.splits = p.splits; a.splits_all = p.splits * p.nseg;
  const bool direct = a.splits_all == 1 && !(vrot && rot != nullptr);
  a.wo = direct ? nullptr : reinterpret_cast<float*>(ws + p.o_o);
  a.wl = direct ? nullptr : reinterpret_cast<float*>(ws + p.o_l);
  a.out = out; a.ot = ot; a.rot = vrot ? ROT_PLAIN : ROT_NONE; a.signs = nullptr;
  a.vscale = raw ? 1.f / v_lift(true, vb) : 32.f / v_lift(false, vb);
  a.oscale = vrot ? fwht_scale(D) : 1.f;
  a.lens = nullptr; a.lens_less = 0; a.hkv_b = hkv;
  a.o_batch = 0; a.o_row = o_row; a.o_head = o_head;
  const V1Geom geo = raw ? V1Geom{2 * D, 2 * D, 2 * D, 4 * D} : v1_geom(D, kb, vb, (flags & V1F_KFP8) != 0);
  const int wide = (((uintptr_t)cache | (uintptr_t)sblk | (uintptr_t)spos | (uintptr_t)shead) & 15) == 0;  // 16-byte slots
  const int pitch = ((geo.raw + 3) / 4 + 1) | 1;  // a pad dword, odd
  for (int s = 0; s < p.nseg; ++s) {
    a.seg0 = p.base + s * p.seg;
    a.seg1 = std::min(a.seg0 + p.seg, total);
    a.split0 = s * p.splits;
    // whole 64-token tiles: positions past the sequence are written as hidden
    const int tiles = (a.seg1 - a.seg0 + 63) / 64 * 2;
    chunk_gather_v1_kernel<D, KHL><<<dim3(tiles, hkv), dim3(256), (size_t)pitch * 32 * 4, st>>>(
        cache, nb, lbs, sblk, spos, shead, bt, mb, cent, kb, vb, (flags & V1F_KFP8) != 0, a.seg0, total, pitch, wide, kf,
        p.kstride, vf, p.vstride, tok, p.tstride);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    chunk_attn_kernel<D, 2, KHL, false, true><<<dim3((unsigned)(hkv * (p.colpad / p.cols)), p.splits), dim3(256), 0, st>>>(a);
    if ((e = hipGetLastError()) != hipSuccess) return e;
  }
  if (direct) return hipSuccess;
  const int64_t mrows = (int64_t)nq * hq;
  const float rs = fwht_scale(D);
#define FTQ_CHUNK_MERGE(R, S, F)                                                                                  \
  return ot == F32   ? launch_merge_splits<D, F32, R>(a.wo, a.wl, mrows, a.splits_all, S, F, out, st)           \
         : ot == F16 ? launch_merge_splits<D, F16, R>(a.wo, a.wl, mrows, a.splits_all, S, F, out, st)           \
                     : launch_merge_splits<D, BF16, R>(a.wo, a.wl, mrows, a.splits_all, S, F, out, st)
  if (vrot && rot != nullptr) FTQ_CHUNK_MERGE(ROT_MATRIX, rot, 1.f);
  if (vrot) FTQ_CHUNK_MERGE(ROT_PLAIN, nullptr, rs);
  FTQ_CHUNK_MERGE(ROT_NONE, nullptr, rs);
#undef FTQ_CHUNK_MERGE
}

}  // namespace
}  // namespace ftq

using namespace ftq;

extern "C" int64_t ftq_v1_chunk_workspace_bytes(int n_query, int num_q_heads, int num_kv_heads, int d, int past_len,
                                                int key_bits, int value_bits, int v_flags, int window) {
  ChunkPlan p;
  if (!(d == 64 || d == 128 || d == 256) ||
      !(key_bits == KB_RAW ? value_bits == KB_RAW : v1_widths_ok(key_bits, value_bits, v_flags)) ||
      !chunk_plan(p, n_query, num_q_heads, num_kv_heads, d, past_len, key_bits, value_bits, v_flags, window, true))
    return -1;
  return p.bytes;
}

extern "C" int ftq_v1_chunk_attention(const void* query, int q_dtype, const uint8_t* kv_cache, int64_t num_blocks,
                                      int block_size, int64_t stride_block, int64_t stride_pos, int64_t stride_head,
                                      const int32_t* block_row, int max_blocks, int past_len, int n_query,
                                      int num_q_heads, int num_kv_heads, int d, const float* centroids, int key_bits,
                                      int value_bits, float scale, int v_flags, int window, void* workspace,
                                      int64_t workspace_bytes, void* out, int out_dtype, const float* rotation,
                                      void* stream) {
  const bool raw = key_bits == KB_RAW;
  FTQ_REQUIRE(d == 64 || d == 128 || d == 256, "chunk attention: head_dim must be 64, 128 or 256");
  FTQ_REQUIRE(raw ? (value_bits == KB_RAW && v_flags == 0 && rotation == nullptr)
                  : v1_widths_ok(key_bits, value_bits, v_flags),
              "chunk attention: key_bits and value_bits must both be in 1..4, both 8 or both 16 (raw fp16 slots, no flags)");
  FTQ_REQUIRE((v_flags & ~(V1F_VROT | V1F_KFP8)) == 0, "chunk attention: v_flags bits 0 (V rotated) and 2 (fp8 keys) only");
  FTQ_REQUIRE(block_size >= 16 && block_size <= 4096 && (block_size & (block_size - 1)) == 0,
              "block_size must be a power of two in [16, 4096]");
  FTQ_REQUIRE(n_query >= 0 && past_len >= 0 && num_kv_heads > 0 && num_q_heads > 0 && num_blocks >= 0 && max_blocks >= 0,
              "bad token / head / block counts");
  FTQ_REQUIRE(num_q_heads % num_kv_heads == 0, "num_q_heads must be a multiple of num_kv_heads");
  FTQ_REQUIRE(num_q_heads / num_kv_heads <= 16, "GQA group (num_q_heads / num_kv_heads) must be <= 16");
  FTQ_REQUIRE(window >= 0, "window must be >= 0 (0: none)");
  FTQ_REQUIRE(q_dtype >= F32 && q_dtype <= BF16 && out_dtype >= F32 && out_dtype <= BF16,
              "dtype must be FTQ_F32, FTQ_F16 or FTQ_BF16");
  const int raw_bytes = raw ? 4 * d : v1_geom(d, key_bits, value_bits, (v_flags & V1F_KFP8) != 0).raw;
  FTQ_REQUIRE(stride_head >= raw_bytes, "stride_head is smaller than the slot bytes");
  FTQ_REQUIRE(cache_strides_ok(num_blocks, stride_block, stride_pos, stride_head, num_kv_heads, block_size),
              "kv_cache strides must describe [num_blocks][block_size][num_kv_heads][slot]");
  FTQ_REQUIRE(stride_head % 4 == 0 && stride_pos % 4 == 0 && stride_block % 4 == 0,
              "kv_cache strides must be multiples of 4 bytes");
  if (n_query == 0) return FTQ_OK;
  FTQ_REQUIRE(num_blocks >= 1, "kv_cache must hold at least one block");
  FTQ_REQUIRE(query && kv_cache && block_row && out && workspace, "null pointer argument");
  FTQ_REQUIRE(centroids != nullptr || raw || (v_flags & V1F_KFP8) != 0, "null centroids");
  FTQ_REQUIRE(aligned16(query) && aligned16(out) && aligned16(workspace) && aligned4(kv_cache),
              "query, out and workspace must be 16-byte aligned, kv_cache 4-byte aligned");
  FTQ_REQUIRE(rotation == nullptr || aligned4(rotation), "rotation must be 4-byte aligned");
  ChunkPlan p;
  FTQ_REQUIRE(chunk_plan(p, n_query, num_q_heads, num_kv_heads, d, past_len, key_bits, value_bits, v_flags, window,
                         rotation != nullptr && (v_flags & V1F_VROT) != 0),
              "chunk attention: too many tokens");
  FTQ_REQUIRE(workspace_bytes >= p.bytes, "workspace too small (see ftq_v1_chunk_workspace_bytes)");
  FTQ_REQUIRE((int64_t)num_kv_heads * (p.colpad / p.cols) <= INT32_MAX && num_kv_heads <= 65535, "grid too large");
  int lbs = 0;
  while ((1 << lbs) < block_size) ++lbs;
  uint8_t* ws = static_cast<uint8_t*>(workspace);
  hipStream_t st = (hipStream_t)stream;
  const int64_t row = (int64_t)num_q_heads * d;
#define FTQ_CHUNK_GO(D, KHL)                                                                                          \
  chunk_launch<D, KHL>(p, query, q_dtype, row, D, kv_cache, num_blocks, lbs, stride_block, stride_pos, stride_head,   \
                       block_row, max_blocks, past_len, n_query, num_q_heads, num_kv_heads, centroids, key_bits,      \
                       value_bits, v_flags, scale, window, ws, out, out_dtype, row, D, rotation, st)
  hipError_t e;
  if (d == 64) e = FTQ_CHUNK_GO(64, true);
  else if (d == 256) e = FTQ_CHUNK_GO(256, true);
  else if (p.khl) e = FTQ_CHUNK_GO(128, true);
  else e = FTQ_CHUNK_GO(128, false);
#undef FTQ_CHUNK_GO
  return hip_status(e);
}
