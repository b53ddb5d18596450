// vLLM v1 slot decode attention at float32-level products on the matrix cores,
// for head_dim 64 and 256 with 2-4 bit keys and 2-4 bit uniform values (the
// semantics of ftq_v1.hip; reference vllm_plugin/triton_decode_offset.py:42-442).
//
// Every operand that is not exact in f16 enters as hi + lo (x = hi + lo to
// 2^-22 relative): the K table values (scaled by a power of two), the rotated
// query (scaled per head), and the softmax weights times the V scale.  Sums
// are fp32, the low products summed apart.  The V codes are exact: centred
// (code - mid) 2^e, with e the token's own scale exponent and mid's share of
// the sum moved to the minimum, so that no offset has to cancel.  Relative
// error against 64 bits over 14 shapes, unit-normal queries: 1.4e-7 to 4.4e-7,
// the fp32 FMA kernel (ftq_v1_valu.hip, which stays for the other formats and
// on request) 3.2e-7 to 3.3e-6; queries 6 times larger: 3e-7 to 1.5e-6 in both.
//
// What the FMA kernel is bound by: one LDS read of four query values and five
// FMAs per K element (24 sequences x 8 kv heads, 700-6000 positions, d = 64,
// K4 V4, group 4: 57 us; d = 256: 160 us for 2 x 4 heads at 5120 positions).
// Here the products are MFMAs and what is left per K element is half a table
// lookup: the same call at d = 64 takes 37 us (HBM traffic of its 128-byte
// slots: 17 us), 64 x 8 units of 2048-2304 positions at K3 V3 86 -> 48 us;
// d = 256, 16 x 8 units of 4000 positions, K3 V3, 451 -> 62 us.
//
// One workgroup (4 waves) per (batch, kv head, split); a wave takes every 4th
// 32-token tile (two 16-token S-tiles).
//   S^T = K Q^T: A = K pairs (hi, then lo) from an LDS table of 8-byte
//     entries, B = the query, column h its hi part and column 8 + h its lo part
//     (QL: more than 8 heads, lo as a second operand).
//   ||c||^2: Gram diagonal, hi hi + 2 lo hi.
//   O^T = V^T P^T: A = V codes of the lane's 8 tokens, B = P', hi in column h
//     and lo in column 8 + h (QL: a second operand), one accumulator column
//     each, added after the last tile.
#include "ftq_attn_dev.h"
#include "ftq_internal.h"
#include "ftq_merge.h"
#include "ftq_v1_dev.h"

#include <algorithm>
#include <cmath>

namespace ftq {

float fwht_scale(int d);

namespace {

struct __attribute__((packed, aligned(2))) U32x2B { uint32_t v; };
struct __attribute__((packed, aligned(2))) U64x2B { uint64_t v; };
typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));

template <int D, int KB, int VB>
struct SGeo {
  static constexpr V1Geom G = v1_geom(D, KB, VB);
  static constexpr int KQ = D * KB / 32;         // K bytes of one lane (a quarter of a vector)
  static constexpr int KW = (KQ + 3) / 4;        // ... in dwords
  static constexpr int NS = D / 32, NB = D / 16;
  static constexpr int VBITS = NB * VB;          // V code bits of one lane and token: dims [NB m, NB m + NB)
  static constexpr bool VSH = VBITS % 16 != 0;   // they start inside a 16-bit unit
  // dwords loaded per token from the even byte at or below the lane's first bit
  static constexpr int VW = (VBITS + (VSH ? 12 : 0) + 31) / 32;
  static constexpr int DPC = 16 / VB;            // dims whose codes one 16-bit window holds
  static constexpr int NCH = (NB + DPC - 1) / DPC;
  static constexpr int LOGC = 4;                 // table copies: 16 (a phase of 16 lanes reads 8 bytes each)
  static constexpr int ENTRIES = 1 << (2 * KB);
  static constexpr int TAB_BYTES = ENTRIES * 8 << LOGC;
};

template <int D, int KB, int VB>
struct STile {
  using Q = SGeo<D, KB, VB>;
  uint32_t k[2][Q::KW];
  uint32_t v[2][4][Q::VW];
  uint32_t kn[2], vs[2], vm[2];  // f16 bits of token m's K norm, V scale, V min
  bool ok[2];
};

// NB bytes at an even offset, into (NB + 3) / 4 dwords (a 6-byte field reads
// 8: the slot goes on past its codes)
template <int NB>
__device__ __forceinline__ void load_even(const uint8_t* base, uint32_t off, uint32_t (&w)[(NB + 3) / 4]) {
  const uint8_t* p = base + off;
  if constexpr (NB == 2) {
    w[0] = *reinterpret_cast<const uint16_t*>(p);
  } else if constexpr (NB <= 4) {
    w[0] = reinterpret_cast<const U32x2B*>(p)->v;
  } else {
#pragma unroll
    for (int i = 0; i < (NB + 7) / 8; ++i) {
      const uint64_t x = reinterpret_cast<const U64x2B*>(p + 8 * i)->v;
      w[2 * i] = (uint32_t)x;
      w[2 * i + 1] = (uint32_t)(x >> 32);
    }
  }
}

template <int D, int KB, int VB>
__device__ __forceinline__ void stile_load(STile<D, KB, VB>& r, int st, const uint8_t* cache, int phys, int nb32,
                                           uint32_t within, int64_t s_blk, uint32_t s_pos, int64_t kvh_off,
                                           uint32_t koff, uint32_t toff, uint32_t voff) {
  using Q = SGeo<D, KB, VB>;
  const bool ok = (uint32_t)phys < (uint32_t)nb32;
  // a tile without a page reads block 0 (the loads always issue) and is masked
  const uint8_t* bst = cache + ((int64_t)(ok ? phys : 0) * s_blk + (int64_t)(ok ? within : 0u) * s_pos + kvh_off);
  load_even<Q::KQ>(bst, koff, r.k[st]);
  r.kn[st] = *reinterpret_cast<const uint16_t*>(bst + toff + Q::G.mse);
  r.vs[st] = *reinterpret_cast<const uint16_t*>(bst + toff + Q::G.kps + Q::G.vdb);
  r.vm[st] = *reinterpret_cast<const uint16_t*>(bst + toff + Q::G.kps + Q::G.vdb + 2);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint8_t* tp = bst + (uint32_t)i * s_pos;
    if constexpr (!Q::VSH) load_even<Q::VBITS / 8>(tp, voff, r.v[st][i]);
    else if constexpr (Q::VBITS + 12 <= 16 || VB != 3) load_even<2>(tp, voff, r.v[st][i]);
    else load_even<4>(tp, voff, r.v[st][i]);
  }
  r.ok[st] = ok;
}

// the 16-bit window of dims [DPC c, DPC c + DPC) of two tokens, one per half
template <int VB, int DPC, int N>
__device__ __forceinline__ uint32_t v_window(const uint32_t (&a)[N], const uint32_t (&b)[N], int c) {
  const int bit = c * DPC * VB, w = bit >> 5, o = bit & 31;
  if (o == 0) return __builtin_amdgcn_perm(b[w], a[w], 0x05040100u);
  if (o == 16) return __builtin_amdgcn_perm(b[w], a[w], 0x07060302u);
  const uint32_t x = w + 1 < N ? __builtin_amdgcn_alignbit(a[w + 1], a[w], o) : a[w] >> o;
  const uint32_t y = w + 1 < N ? __builtin_amdgcn_alignbit(b[w + 1], b[w], o) : b[w] >> o;
  return __builtin_amdgcn_perm(y, x, 0x05040100u);
}

__device__ __forceinline__ uint32_t sp_pk_f16(float a, float b) {
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{a, b}), half2_t));
}

template <int D, int KB, int VB, bool QL>
__global__ __launch_bounds__(256, 2) void v1_attn_split_kernel(
    const void* __restrict__ query, int qt, const uint8_t* __restrict__ cache, const int32_t* __restrict__ block_table,
    const int32_t* __restrict__ seq_lens, const int32_t* __restrict__ kv_start, int hq, int hkv, int lbs, int max_blocks,
    int64_t num_blocks, int64_t s_blk, int64_t s_pos, int64_t s_head, const float* __restrict__ cent, float qscale,
    int num_splits, float* __restrict__ ws_o, float* __restrict__ ws_lse, const float* __restrict__ rot, int direct,
    float oscale, void* __restrict__ out, int ot, float* __restrict__ lse) {
  using Q = SGeo<D, KB, VB>;
  constexpr int NS = Q::NS, NB = Q::NB, E = D / 16;
  constexpr int QS_BYTES = 16 * (D + 4) * 4;
  extern __shared__ __attribute__((aligned(16))) uint8_t pool[];  // rotated queries, then the wave merge
  __shared__ __attribute__((aligned(16))) uint2 tab[Q::TAB_BYTES / 8];
  __shared__ __attribute__((aligned(16))) float fields[4][2][4][16];  // [wave][S-tile][K factor, V factor, V offset, 2^e][token]
  __shared__ float red_m[4][16], red_l[4][16], red_z[4][16], qinv[16];
  float (*qs)[D + 4] = reinterpret_cast<float (*)[D + 4]>(pool);
  static_assert(QS_BYTES <= 65536, "query rows");

  const int split = blockIdx.x, kvh = blockIdx.y, b = blockIdx.z;
  const int G = hq / hkv;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int m = lane & 15, g = lane >> 4;
  const int wave_u = __builtin_amdgcn_readfirstlane(wave);

  // ---- the split's tiles, and the first tile's loads ----
  const int seq_len = seq_lens[b];
  int k0 = kv_start ? kv_start[b] : 0;
  if (k0 < 0) k0 = 0;
  const int t_first = k0 >> 5, t_last = (seq_len + 31) >> 5;
  const int n_tiles = t_last > t_first ? t_last - t_first : 0;
  const int tps = (n_tiles + num_splits - 1) / num_splits;
  const int t_begin = t_first + split * tps, t_end = min(t_begin + tps, t_last);
  const int32_t* bt_row = block_table + (int64_t)b * max_blocks;
  const int64_t kvh_off = (int64_t)kvh * s_head;
  const int nb32 = (int)min(num_blocks, (int64_t)0x7fffffff);
  const uint32_t sp32 = (uint32_t)s_pos;
  const uint32_t koff = (uint32_t)m * sp32 + (uint32_t)(g * Q::KQ), toff = (uint32_t)m * sp32;
  constexpr int NBVB = Q::VBITS;
  const uint32_t vbyte = (uint32_t)(NBVB * m >> 3) & ~1u;
  const uint32_t voff = (uint32_t)(4 * g) * sp32 + (uint32_t)Q::G.kps + vbyte;
  const uint32_t vsh = (uint32_t)(NBVB * m) - 8u * vbyte;
  struct Bt { int e[2]; };
  auto bt_of = [&](int t) __attribute__((always_inline)) {  // block-table entries: uniform, one tile ahead of their loads
    Bt r;
#pragma unroll
    for (int st = 0; st < 2; ++st) {
      const int pos0 = t * 32 + st * 16, page = pos0 >> lbs;
      r.e[st] = (t < t_end && pos0 < seq_len && page < max_blocks) ? bt_row[page] : -1;
    }
    return r;
  };
  auto load = [&](STile<D, KB, VB>& r, Bt bt, int t) __attribute__((always_inline)) {
#pragma unroll
    for (int st = 0; st < 2; ++st)
      stile_load(r, st, cache, bt.e[st], nb32, (uint32_t)((t * 32 + st * 16) & ((1 << lbs) - 1)), s_blk, sp32, kvh_off, koff,
                 toff, voff);
  };
  STile<D, KB, VB> ra, rb;
  int tile = t_begin + wave_u;
  Bt btn{{-1, -1}};
  if (tile < t_end) {
    load(ra, bt_of(tile), tile);
    btn = bt_of(tile + 4);
  }

  // ---- prologue: queries (one head per 16 lanes) and the K table ----
  {
    const int hh = tid >> 4, l16 = tid & 15;
    if (hh < G) {
      float y[E];
      const int64_t off = ((int64_t)b * hq + kvh * G + hh) * D + l16 * E;
      if (qt == F32) load_elems<F32, E>(query, off, y);
      else if (qt == F16) load_elems<F16, E>(query, off, y);
      else load_elems<BF16, E>(query, off, y);
      if (rot != nullptr) rot_matrix_lanes<D, E>(y, rot, &qs[hh][0], l16);
      else fwht_lanes<E, 16>(y, l16);
      // each head scaled by the power of two that puts its largest magnitude in
      // [256, 512): the low parts of the others stay normal f16 numbers
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
      const int ue = min(max(135 + 127 - (int)((__float_as_uint(mx) >> 23) & 255u), 1), 253);
      const float up = __uint_as_float((uint32_t)ue << 23);
      if (l16 == 0) qinv[hh] = __uint_as_float((uint32_t)(254 - ue) << 23);
#pragma unroll
      for (int i = 0; i < E; ++i) qs[hh][l16 * E + i] = y[i] * up;
    } else if (hh < 16 && l16 == 0) {
      qinv[hh] = 0.f;
    }
  }
  float tsc_inv;
  {  // levels times the power of two that puts the largest in [512, 1024), as hi + lo pairs
    constexpr int NL = 1 << KB;
    float mx = 0.f;
#pragma unroll
    for (int i = 0; i < NL; ++i) mx = fmaxf(mx, fabsf(cent[i]));
    const bool fin = mx > 0.f && mx < INFINITY;
    const int ue = fin ? min(max(263 - (int)((__float_as_uint(mx) >> 23) & 255u), 1), 253) : 127;
    const float sc = __uint_as_float((uint32_t)ue << 23);
    tsc_inv = __uint_as_float((uint32_t)(254 - ue) << 23);
    // a thread's entry is fixed (ENTRIES divides 256): its two levels are read
    // once, and its copies written two at a time, in an order that starts at
    // the entry, so that a wave's writes spread over the banks
    const int c = tid & (Q::ENTRIES - 1);
    const float x = sc * cent[c & (NL - 1)], y = sc * cent[c >> KB];
    const uint32_t h = sp_pk_f16(x, y);
    const half2_t hv = __builtin_bit_cast(half2_t, h);
    const uint32_t l = sp_pk_f16(x - (float)hv[0], y - (float)hv[1]);
#pragma unroll
    for (int i = 0; i < (Q::ENTRIES * 8 + 255) / 256; ++i) {
      const int k = (i * 256 + tid) / Q::ENTRIES;  // pair of copies
      if (k < 8) *reinterpret_cast<uint4*>(&tab[(c << Q::LOGC) + 2 * ((k + c) & 7)]) = make_uint4(h, l, h, l);
    }
  }
  __syncthreads();
  const uint32_t laneoff = 8u * (uint32_t)(lane & 15);
  Op8 qb[NS], ql[QL ? NS : 1];
  {
    const int hh = (!QL && m >= 8) ? m - 8 : m;
    const bool lo_col = hh != m;
#pragma unroll
    for (int s = 0; s < NS; ++s)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        float x = 0.f, y = 0.f;
        if (hh < G) {
          x = qs[hh][g * (D / 4) + 8 * s + 2 * j];
          y = qs[hh][g * (D / 4) + 8 * s + 2 * j + 1];
        }
        const uint32_t h = sp_pk_f16(x, y);
        const half2_t hv = __builtin_bit_cast(half2_t, h);
        const uint32_t l = sp_pk_f16(x - (float)hv[0], y - (float)hv[1]);
        qb[s].u[j] = lo_col ? l : h;
        if constexpr (QL) ql[s].u[j] = l;
      }
  }
  const float qf = qinv[(!QL && m >= 8) ? m - 8 : m] * tsc_inv;  // of the lane's column (head)

  constexpr float V_LIFT = 32.f, TAU = 4.f, MINF = -3.0e38f, MID = 0.5f * (float)((1 << VB) - 1);
  float m_run = MINF, l_run = 0.f, z_run = 0.f;
  floatx4 acc[NB];
#pragma unroll
  for (int i = 0; i < NB; ++i) acc[i] = floatx4{0.f, 0.f, 0.f, 0.f};

  auto process = [&](const STile<D, KB, VB>& cur, int t) __attribute__((always_inline)) {
    floatx4 s[2];
    __asm__ volatile("" ::: "memory");  // a wave's LDS accesses run in order
#pragma unroll
    for (int st = 0; st < 2; ++st) {
      floatx4 c = {0.f, 0.f, 0.f, 0.f}, cl = c, g1 = c, g2 = c;
#pragma unroll
      for (int i = 0; i < NS; ++i) {
        Op8 h, l;
#pragma unroll
        for (int p = 0; p < 4; ++p) {
          const uint2 e = *reinterpret_cast<const uint2*>(reinterpret_cast<const uint8_t*>(tab) +
                                                          lut_field<3 + Q::LOGC, 2 * KB>(cur.k[st], (8 * i + 2 * p) * KB, laneoff));
          h.u[p] = e.x;
          l.u[p] = e.y;
        }
        c = __builtin_amdgcn_mfma_f32_16x16x32_f16(h.h, qb[i].h, c, 0, 0, 0);
        cl = __builtin_amdgcn_mfma_f32_16x16x32_f16(l.h, qb[i].h, cl, 0, 0, 0);
        g1 = __builtin_amdgcn_mfma_f32_16x16x32_f16(h.h, h.h, g1, 0, 0, 0);
        g2 = __builtin_amdgcn_mfma_f32_16x16x32_f16(l.h, h.h, g2, 0, 0, 0);
        if constexpr (QL) cl = __builtin_amdgcn_mfma_f32_16x16x32_f16(h.h, ql[i].h, cl, 0, 0, 0);
      }
      // token m: sum c^2 from the diagonal (rows 4g + i, column m), K and V factors
      const int i3 = m & 3;
      const float d1 = i3 == 0 ? g1[0] : i3 == 1 ? g1[1] : i3 == 2 ? g1[2] : g1[3];
      const float d2 = i3 == 0 ? g2[0] : i3 == 1 ? g2[1] : i3 == 2 ? g2[2] : g2[3];
      const float csq = warp_sum_q((m >> 2) == g ? __builtin_fmaf(2.f, d2, d1) : 0.f) * (tsc_inv * tsc_inv);
      const float kn = (float)__builtin_bit_cast(_Float16, (uint16_t)cur.kn[st]);
      const float sc = (float)__builtin_bit_cast(_Float16, (uint16_t)cur.vs[st]);
      const float mn = (float)__builtin_bit_cast(_Float16, (uint16_t)cur.vm[st]);
      // V operand (code - mid) 2^e: 2^(e + 5) the scale's own power of two (its
      // factor in [32, 64) V_LIFT, so that small weights' low parts stay normal:
      // 16 times it is the largest f16), e where codes stay normal and (2^VB +
      // mid) 2^e finite
      const int e = min(max((int)((cur.vs[st] >> 10) & 31u) - 20, -14), 11);
      const float x = g == 0 ? kn / __builtin_sqrtf(csq + 1e-16f)
                    : g == 1 ? sc * (V_LIFT * __uint_as_float((uint32_t)(127 - e) << 23))
                    : g == 2 ? __builtin_fmaf(MID, sc, mn)
                             : __uint_as_float((uint32_t)(127 + e) << 23);
      fields[wave][st][g][m] = x;
      if constexpr (QL) {
        s[st] = c + cl;
      } else {  // columns h and 8 + h: hi and lo products; both columns end with the sum
#pragma unroll
        for (int i = 0; i < 4; ++i) s[st][i] = (c[i] + dpp_xor8(c[i])) + (cl[i] + dpp_xor8(cl[i]));
      }
    }
    __asm__ volatile("" ::: "memory");
    float vf[2][4], vz[2][4], ve[2][4];
#pragma unroll
    for (int st = 0; st < 2; ++st) {
      const float4 k4 = *reinterpret_cast<const float4*>(&fields[wave][st][0][4 * g]);
      const float4 f4 = *reinterpret_cast<const float4*>(&fields[wave][st][1][4 * g]);
      const float4 z4 = *reinterpret_cast<const float4*>(&fields[wave][st][2][4 * g]);
      const float4 e4 = *reinterpret_cast<const float4*>(&fields[wave][st][3][4 * g]);
      const float ka[4] = {k4.x, k4.y, k4.z, k4.w};
      vf[st][0] = f4.x; vf[st][1] = f4.y; vf[st][2] = f4.z; vf[st][3] = f4.w;
      vz[st][0] = z4.x; vz[st][1] = z4.y; vz[st][2] = z4.z; vz[st][3] = z4.w;
      ve[st][0] = e4.x; ve[st][1] = e4.y; ve[st][2] = e4.z; ve[st][3] = e4.w;
#pragma unroll
      for (int i = 0; i < 4; ++i) s[st][i] = s[st][i] * qf * ka[i];
    }
    if (t * 32 < k0 || t * 32 + 32 > seq_len || !cur.ok[0] || !cur.ok[1]) {  // edges; their fields may hold anything
#pragma unroll
      for (int st = 0; st < 2; ++st)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int pos = t * 32 + st * 16 + 4 * g + i;
          if (pos >= seq_len || pos < k0 || !cur.ok[st]) {
            s[st][i] = -INFINITY;
            vf[st][i] = 0.f;
            vz[st][i] = 0.f;
          }
        }
    }
    float tm = fmaxf(fmaxf(fmaxf(s[0][0], s[0][1]), fmaxf(s[0][2], s[0][3])),
                     fmaxf(fmaxf(s[1][0], s[1][1]), fmaxf(s[1][2], s[1][3])));
    tm = warp_max_q(tm);
    if (__builtin_amdgcn_ballot_w64(tm > m_run + TAU) != 0) {  // wave-uniform, rare
      const float mnew = fmaxf(m_run, tm);
      const float al = __builtin_amdgcn_exp2f(m_run - mnew);
      m_run = mnew;
      l_run *= al;
      z_run *= al;
#pragma unroll
      for (int bb = 0; bb < NB; ++bb) acc[bb] *= al;
    }
    // weights: hi in columns h, lo in columns 8 + h (QL: lo as an operand of its own)
    Op8 pb, pl;
    half2_t e2[4], c2[4];  // 2^(e + VB) and -(2^VB + mid) 2^e of the operand pairs' tokens
    const bool lo_col = !QL && m >= 8;
    float lt = 0.f, zt = 0.f;  // the tile's sums first: many small weights beside a large one count
#pragma unroll
    for (int st = 0; st < 2; ++st) {
      float w[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float p = __builtin_amdgcn_exp2f(s[st][i] - m_run);
        lt += p;
        zt = __builtin_fmaf(p, vz[st][i], zt);
        w[i] = p * vf[st][i];
      }
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const uint32_t hi = sp_pk_f16(w[2 * h], w[2 * h + 1]);
        const half2_t hv = __builtin_bit_cast(half2_t, hi);
        const uint32_t lo = sp_pk_f16(w[2 * h] - (float)hv[0], w[2 * h + 1] - (float)hv[1]);
        pb.u[2 * st + h] = lo_col ? lo : hi;
        if constexpr (QL) pl.u[2 * st + h] = lo;
        const half2_t ex = __builtin_bit_cast(half2_t, sp_pk_f16(ve[st][2 * h], ve[st][2 * h + 1]));
        e2[2 * st + h] = ex * (_Float16)(float)(1 << VB);
        c2[2 * st + h] = ex * (_Float16)(-((float)(1 << VB) + MID));
      }
    }
    l_run += lt;
    z_run += zt;
    constexpr uint32_t CM = ((1u << VB) - 1u) << (10 - VB);
#pragma unroll
    for (int ch = 0; ch < Q::NCH; ++ch) {
      uint32_t x[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int st = j >> 1, i = 2 * (j & 1);
        if constexpr (Q::VSH) {
          const uint32_t a[1] = {cur.v[st][i][0] >> vsh}, c[1] = {cur.v[st][i + 1][0] >> vsh};
          x[j] = v_window<VB, Q::DPC>(a, c, ch);
        } else {
          x[j] = v_window<VB, Q::DPC>(cur.v[st][i], cur.v[st][i + 1], ch);
        }
      }
#pragma unroll
      for (int q = 0; q < Q::DPC; ++q) {
        const int bb = ch * Q::DPC + q;
        if (bb < NB) {
          Op8 a;
          const int sh = 10 - VB - q * VB;  // the code's bits to the top of the f16 mantissa: 1 + code 2^-VB
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const uint32_t y = ((sh >= 0 ? x[j] << sh : x[j] >> -sh) & (CM * 0x10001u)) | 0x3C003C00u;
            const half2_t v = __builtin_elementwise_fma(__builtin_bit_cast(half2_t, y), e2[j], c2[j]);
            a.u[j] = __builtin_bit_cast(uint32_t, v);
          }
          acc[bb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a.h, pb.h, acc[bb], 0, 0, 0);
          if constexpr (QL) acc[bb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a.h, pl.h, acc[bb], 0, 0, 0);
        }
      }
    }
  };

  // a fixed assignment of tiles, so that the sums do not depend on how fast
  // the waves progress; block-table entries two tiles ahead
  while (tile < t_end) {
    Bt nx = bt_of(tile + 8);
    load(rb, btn, tile + 4);
    btn = nx;
    process(ra, tile);
    tile += 4;
    if (tile >= t_end) break;
    nx = bt_of(tile + 8);
    load(ra, btn, tile + 4);
    btn = nx;
    process(rb, tile);
    tile += 4;
  }

  // ---- the 4 waves meet in LDS (the pool of the rotated queries) ----
  __syncthreads();
  const float l_tot = warp_sum_q(l_run), z_tot = warp_sum_q(z_run);
  if (g == 0) {
    red_m[wave][m] = m_run;
    red_l[wave][m] = l_tot;
    red_z[wave][m] = z_tot;
  }
  float* red_o = reinterpret_cast<float*>(pool);  // [4][G][D + 1]
#pragma unroll
  for (int bb = 0; bb < NB; ++bb)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      // row 4g + i of accumulator bb is dim NB (4g + i) + bb
      const float o = (QL ? acc[bb][i] : acc[bb][i] + dpp_xor8(acc[bb][i])) * (1.f / V_LIFT);
      if (m < G) red_o[(wave * G + m) * (D + 1) + NB * (4 * g + i) + bb] = o;
    }
  __syncthreads();
  constexpr int E2 = D / 64;
  for (int h = wave; h < G; h += 4) {
    float M = MINF;
#pragma unroll
    for (int w = 0; w < 4; ++w) M = fmaxf(M, red_m[w][h]);
    float L = 0.f, o[E2];
#pragma unroll
    for (int i = 0; i < E2; ++i) o[i] = 0.f;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const float f = red_m[w][h] == MINF ? 0.f : __builtin_amdgcn_exp2f(red_m[w][h] - M);
      if (f != 0.f) {
        L += f * red_l[w][h];
#pragma unroll
        for (int i = 0; i < E2; ++i) o[i] += f * (red_o[(w * G + h) * (D + 1) + E2 * lane + i] + red_z[w][h]);
      }
    }
#pragma unroll
    for (int i = 0; i < E2; ++i) o[i] = L > 0.f ? o[i] / L : 0.f;
    const int64_t row = (int64_t)b * hq + kvh * G + h;
    if (direct < 0) {
      float* dst = ws_o + (row * num_splits + split) * D + E2 * lane;
#pragma unroll
      for (int i = 0; i < E2; ++i) dst[i] = o[i];
      if (lane == 0) ws_lse[row * num_splits + split] = L > 0.f ? M + __builtin_log2f(L) : -INFINITY;
      continue;
    }
    if (direct == 1) {
      fwht_wave64<E2>(o, lane);
#pragma unroll
      for (int i = 0; i < E2; ++i) o[i] *= oscale;
    }
    if (lse != nullptr && lane == 0) lse[row] = L > 0.f ? (M + __builtin_log2f(L)) * 0.69314718055994531f : -INFINITY;
    if (ot == F32) store_small<F32, E2>(out, row * D + lane * E2, o);
    else if (ot == F16) store_small<F16, E2>(out, row * D + lane * E2, o);
    else store_small<BF16, E2>(out, row * D + lane * E2, o);
  }
}

template <int D>
size_t split_lds(int G) {
  return std::max((size_t)16 * (D + 4) * 4, (size_t)4 * G * (D + 1) * 4);
}

template <int D, int KB, int VB, bool QL>
hipError_t split_launch(const V1Args& a, hipStream_t st) {
  const bool direct = a.splits == 1 && !((a.vrot & V1F_VROT) && a.rot != nullptr);
  v1_attn_split_kernel<D, KB, VB, QL><<<dim3(a.splits, a.hkv, a.B), dim3(256), split_lds<D>(a.hq / a.hkv), st>>>(
      a.q, a.qt, a.cache, a.bt, a.sl, a.ks, a.hq, a.hkv, a.lbs, a.max_blocks, a.nb, a.sblk, a.spos, a.shead, a.cent,
      a.qscale, a.splits, a.wo, a.wl, a.rot, direct ? (a.vrot & V1F_VROT) : -1, fwht_scale(D), a.out, a.ot, a.lse);
  return hipGetLastError();
}

template <int D, int KB, int VB>
hipError_t split_launch_g(const V1Args& a, hipStream_t st) {
  return a.hq / a.hkv > 8 ? split_launch<D, KB, VB, true>(a, st) : split_launch<D, KB, VB, false>(a, st);
}
template <int D, int KB>
hipError_t split_launch_v(int vb, const V1Args& a, hipStream_t st) {
  if (vb == 2) return split_launch_g<D, KB, 2>(a, st);
  if (vb == 3) return split_launch_g<D, KB, 3>(a, st);
  return split_launch_g<D, KB, 4>(a, st);
}
template <int D>
hipError_t split_launch_k(int kb, int vb, const V1Args& a, hipStream_t st) {
  if (kb == 2) return split_launch_v<D, 2>(vb, a, st);
  if (kb == 3) return split_launch_v<D, 3>(vb, a, st);
  return split_launch_v<D, 4>(vb, a, st);
}

template <int D>
hipError_t split_merge(const V1Args& a, hipStream_t st) {
  const int64_t rows = (int64_t)a.B * a.hq;
  const float rs = fwht_scale(D);
#define FTQ_SPLIT_MERGE(R, S, F)                                                                                   \
  return a.ot == F32   ? launch_merge_splits<D, F32, R>(a.wo, a.wl, rows, a.splits, S, F, a.out, st, a.lse)      \
         : a.ot == F16 ? launch_merge_splits<D, F16, R>(a.wo, a.wl, rows, a.splits, S, F, a.out, st, a.lse)      \
                       : launch_merge_splits<D, BF16, R>(a.wo, a.wl, rows, a.splits, S, F, a.out, st, a.lse)
  if ((a.vrot & V1F_VROT) && a.rot != nullptr) FTQ_SPLIT_MERGE(ROT_MATRIX, a.rot, 1.f);
  if (a.vrot & V1F_VROT) FTQ_SPLIT_MERGE(ROT_PLAIN, nullptr, rs);
  FTQ_SPLIT_MERGE(ROT_NONE, nullptr, rs);
#undef FTQ_SPLIT_MERGE
}

}  // namespace

// 1-bit codes stay on the FMA kernel: their errors against 64 bits were larger
// here (d = 64, K1 V1, outlier keys: 3.9e-7 against 1.3e-7).
bool v1_split_takes(int d, int kb, int vb, int flags) {
  return (d == 64 || d == 256) && kb >= 2 && kb <= 4 && vb >= 2 && vb <= 4 && (flags & (V1F_KFP8 | V1F_FP32)) == 0 &&
         !((flags & V1F_VLM) != 0 && vb == 4);
}

hipError_t v1_split_launch(const V1Args& a, int d, int kb, int vb, hipStream_t st) {
  hipError_t e = d == 64 ? split_launch_k<64>(kb, vb, a, st) : split_launch_k<256>(kb, vb, a, st);
  if (e != hipSuccess || (a.splits == 1 && !((a.vrot & V1F_VROT) && a.rot != nullptr))) return e;
  return d == 64 ? split_merge<64>(a, st) : split_merge<256>(a, st);
}

// Workgroups of the kernel for 4-bit codes that the GPU holds at once.
int v1_split_resident(int d) {
  if (d == 64) {
    static const int c = resident_workgroups(v1_attn_split_kernel<64, 4, 4, false>);
    return c;
  }
  static const int c = resident_workgroups(v1_attn_split_kernel<256, 4, 4, false>);
  return c;
}

}  // namespace ftq
