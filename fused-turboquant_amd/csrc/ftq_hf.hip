// The small per-layer steps around the compressed cache's kernels in the
// HuggingFace attention forward (reference hf/fused_cache.py:195-222, :540-575),
// each one launch where torch ops take ten: the rotary embedding of q and k,
// and the page slots of a step's tokens.
#include "ftq_device.h"
#include "ftq_internal.h"

#include <algorithm>

namespace ftq {
namespace {

struct RopeSide {
  const void* x;
  void* out;                                    // [batch][tokens][heads][d], contiguous
  int64_t s_batch, s_head, s_tok;               // elements
  int heads;
};

// x rounded to the tensor's type and back
template <int DT>
__device__ __forceinline__ float as_type(float x) {
  if constexpr (DT == BF16) return bf16_bits_to_f32(f32_to_bf16_bits(x));
  else if constexpr (DT == F16) return f16_bits_to_f32(f32_to_f16_bits(x));
  else return x;
}

// out = x cos + rotate_half(x) sin, each product and the sum rounded to the
// type (the torch expression's roundings).  A thread takes 8 elements of the
// first half and the 8 that pair with them.  Bound by its launch at a decode
// step and by memory at a prompt.
template <int DT>
__global__ __launch_bounds__(256) void rope_kernel(RopeSide q, RopeSide k, const void* __restrict__ cos,
                                                   const void* __restrict__ sin, int64_t cs_batch, int64_t cs_tok,
                                                   int64_t sn_batch, int64_t sn_tok, int batch, int tokens, int d) {
  const int per = d / 16, heads = q.heads + k.heads;
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x, rows = (int64_t)batch * tokens * heads;
  const int64_t row = i / per;
  if (row >= rows) return;
  const int e = (int)(i - row * per) * 8;
  const int64_t bt = row / heads;
  int h = (int)(row - bt * heads);
  const int b = (int)(bt / tokens), t = (int)(bt - (int64_t)b * tokens);
  const RopeSide s = h < q.heads ? q : k;
  if (h >= q.heads) h -= q.heads;
  float x1[8], x2[8], c1[8], c2[8], s1[8], s2[8];
  const int64_t xo = b * s.s_batch + h * s.s_head + t * s.s_tok + e;
  load_elems<DT, 8>(s.x, xo, x1);
  load_elems<DT, 8>(s.x, xo + d / 2, x2);
  const int64_t co = b * cs_batch + t * cs_tok + e, so = b * sn_batch + t * sn_tok + e;
  load_elems<DT, 8>(cos, co, c1);
  load_elems<DT, 8>(cos, co + d / 2, c2);
  load_elems<DT, 8>(sin, so, s1);
  load_elems<DT, 8>(sin, so + d / 2, s2);
  float y1[8], y2[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    y1[j] = as_type<DT>(x1[j] * c1[j]) + as_type<DT>(-x2[j] * s1[j]);
    y2[j] = as_type<DT>(x2[j] * c2[j]) + as_type<DT>(x1[j] * s2[j]);
  }
  const int64_t oo = (bt * s.heads + h) * d + e;
  store_elems<DT, 8>(s.out, oo, y1);
  store_elems<DT, 8>(s.out, oo + d / 2, y2);
}

// slots[b n + i] = b cap + lens[b] + i, then lens[b] += n; one workgroup per sequence
__global__ __launch_bounds__(256) void append_slots_kernel(int32_t* __restrict__ lens, int64_t* __restrict__ slots, int n,
                                                           int64_t cap) {
  const int b = blockIdx.x;
  const int len = lens[b];
  const int64_t first = (int64_t)b * cap + len;
  for (int i = threadIdx.x; i < n; i += 256) slots[(int64_t)b * n + i] = first + i;
  __syncthreads();  // every thread has read the length
  if (threadIdx.x == 0) lens[b] = len + n;
}

}  // namespace
}  // namespace ftq

using namespace ftq;

extern "C" int ftq_rope(const void* q, void* q_out, int64_t q_batch, int64_t q_head, int64_t q_tok, int num_q_heads,
                        const void* k, void* k_out, int64_t k_batch, int64_t k_head, int64_t k_tok, int num_kv_heads,
                        const void* cos, int64_t cos_batch, int64_t cos_tok, const void* sin, int64_t sin_batch,
                        int64_t sin_tok, int dtype, int batch, int tokens, int d, void* stream) {
  FTQ_REQUIRE(d >= 16 && d % 16 == 0 && d <= 4096, "rope: head_dim must be a multiple of 16");
  FTQ_REQUIRE(batch >= 0 && tokens >= 0 && num_q_heads > 0 && num_kv_heads > 0, "rope: bad counts");
  FTQ_REQUIRE(dtype >= F32 && dtype <= BF16, "dtype must be FTQ_F32, FTQ_F16 or FTQ_BF16");
  if (batch == 0 || tokens == 0) return FTQ_OK;
  FTQ_REQUIRE(q && k && q_out && k_out && cos && sin, "null pointer argument");
  FTQ_REQUIRE(((q_batch | q_head | q_tok | k_batch | k_head | k_tok | cos_batch | cos_tok | sin_batch | sin_tok) & 7) == 0 &&
                  aligned16(q) && aligned16(k) && aligned16(q_out) && aligned16(k_out) && aligned16(cos) && aligned16(sin),
              "rope: rows must be 16-byte aligned");
  const int64_t threads = (int64_t)batch * tokens * (num_q_heads + num_kv_heads) * (d / 16);
  FTQ_REQUIRE((threads + 255) / 256 <= INT32_MAX, "rope: too many rows");
  const dim3 grid((unsigned)((threads + 255) / 256)), block(256);
  const RopeSide a{q, q_out, q_batch, q_head, q_tok, num_q_heads}, b{k, k_out, k_batch, k_head, k_tok, num_kv_heads};
  hipStream_t st = (hipStream_t)stream;
  if (dtype == F32) rope_kernel<F32><<<grid, block, 0, st>>>(a, b, cos, sin, cos_batch, cos_tok, sin_batch, sin_tok, batch, tokens, d);
  else if (dtype == F16) rope_kernel<F16><<<grid, block, 0, st>>>(a, b, cos, sin, cos_batch, cos_tok, sin_batch, sin_tok, batch, tokens, d);
  else rope_kernel<BF16><<<grid, block, 0, st>>>(a, b, cos, sin, cos_batch, cos_tok, sin_batch, sin_tok, batch, tokens, d);
  return hip_status(hipGetLastError());
}

extern "C" int ftq_append_slots(int32_t* lens, int64_t* slots, int batch, int n, int64_t capacity, void* stream) {
  FTQ_REQUIRE(batch >= 0 && n >= 0 && capacity >= 0, "append slots: bad counts");
  if (batch == 0 || n == 0) return FTQ_OK;
  FTQ_REQUIRE(lens && slots, "null pointer argument");
  append_slots_kernel<<<dim3((unsigned)batch), dim3(256), 0, (hipStream_t)stream>>>(lens, slots, n, capacity);
  return hip_status(hipGetLastError());
}
