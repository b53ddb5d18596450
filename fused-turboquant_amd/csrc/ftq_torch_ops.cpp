// PyTorch operator library over the C ABI (include/fused_tq.h): the
// torch.ops.fused_tq.* operators the Python package calls.  Each operator
// checks its tensors with TORCH_CHECK (RuntimeError), takes the current HIP
// stream of the tensors' device, and calls the C entry point; the kernels
// are the ones libfused_tq.so holds.  Schemas mark the tensors an operator
// writes in place (Tensor(a!)); shape-only fake implementations for tracing
// are registered from Python (fused_turboquant/_ops.py).
#include <torch/library.h>
#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>

#include "fused_tq.h"

namespace {

// a rejected argument raises ValueError (as the Python API does), a HIP
// error RuntimeError
void check_rc(int rc) {
  TORCH_CHECK_VALUE(rc != FTQ_ERR_ARG, "fused_tq: ", ftq_last_error());
  TORCH_CHECK(rc == FTQ_OK, "fused_tq: ", ftq_last_error());
}

int dt(const at::Tensor& t) {
  switch (t.scalar_type()) {
    case at::kFloat: return FTQ_F32;
    case at::kHalf: return FTQ_F16;
    case at::kBFloat16: return FTQ_BF16;
    default: TORCH_CHECK(false, "fused_tq: expected float32, float16 or bfloat16, got ", t.scalar_type());
  }
  return FTQ_F32;
}

int dt_of(c10::ScalarType s) {
  switch (s) {
    case at::kFloat: return FTQ_F32;
    case at::kHalf: return FTQ_F16;
    case at::kBFloat16: return FTQ_BF16;
    default: TORCH_CHECK(false, "fused_tq: output dtype must be float32, float16 or bfloat16");
  }
  return FTQ_F32;
}

void on_device(const at::Tensor& t, const char* name) {
  TORCH_CHECK(t.is_cuda(), "fused_tq: ", name, " must be on a ROCm device");
}

void contig(const at::Tensor& t, const char* name) {
  on_device(t, name);
  TORCH_CHECK(t.is_contiguous(), "fused_tq: ", name, " must be contiguous");
}

// t with rows that kernels can read in 16-byte steps: itself, or an aligned copy
// (contiguous() returns a contiguous view at any storage offset as it is)
at::Tensor rows16(const at::Tensor& t) {
  bool ok = t.dim() > 0 && t.stride(-1) == 1 && (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15) == 0;
  for (int64_t i = 0; ok && i + 1 < t.dim(); ++i) ok = t.stride(i) % 8 == 0;
  return ok ? t : t.clone(at::MemoryFormat::Contiguous);
}

void* stream_of(const at::Tensor& t) {
  return (void*)c10::hip::getCurrentHIPStream(t.device().index()).stream();
}

// ---- library-format codec ----------------------------------------------

std::tuple<at::Tensor, at::Tensor> encode(const at::Tensor& x, const at::Tensor& signs, const at::Tensor& boundaries,
                                          int64_t bits, int64_t codebook_class) {
  contig(x, "x");
  contig(signs, "signs");
  contig(boundaries, "boundaries");
  const c10::DeviceGuard g(x.device());
  const int64_t d = x.size(-1);
  const int64_t n = d > 0 ? x.numel() / d : 0;
  auto sizes = x.sizes().vec();
  sizes.back() = d * bits / 8;
  at::Tensor packed = at::empty(sizes, x.options().dtype(at::kByte));
  sizes.pop_back();
  at::Tensor norms = at::empty(sizes, x.options().dtype(at::kHalf));
  check_rc(ftq_encode_cb(x.data_ptr(), dt(x), n, (int)d, signs.data_ptr<float>(), boundaries.data_ptr<float>(),
                         (int)bits, (int)codebook_class, packed.data_ptr<uint8_t>(),
                         reinterpret_cast<uint16_t*>(norms.data_ptr()), stream_of(x)));
  return {packed, norms};
}

std::tuple<at::Tensor, at::Tensor, at::Tensor, at::Tensor> encode_kv(const at::Tensor& k, const at::Tensor& v,
                                                                     const at::Tensor& signs,
                                                                     const at::Tensor& boundaries, int64_t bits,
                                                                     int64_t codebook_class) {
  contig(k, "k");
  contig(v, "v");
  contig(signs, "signs");
  contig(boundaries, "boundaries");
  TORCH_CHECK(k.sizes() == v.sizes() && k.scalar_type() == v.scalar_type() && k.device() == v.device(),
              "fused_tq: k and v must agree in shape, dtype and device");
  const c10::DeviceGuard g(k.device());
  const int64_t d = k.size(-1);
  const int64_t n = d > 0 ? k.numel() / d : 0;
  auto sizes = k.sizes().vec();
  sizes.back() = d * bits / 8;
  at::Tensor kp = at::empty(sizes, k.options().dtype(at::kByte));
  at::Tensor vp = at::empty(sizes, k.options().dtype(at::kByte));
  sizes.pop_back();
  at::Tensor kn = at::empty(sizes, k.options().dtype(at::kHalf));
  at::Tensor vn = at::empty(sizes, k.options().dtype(at::kHalf));
  check_rc(ftq_encode_kv(k.data_ptr(), v.data_ptr(), dt(k), n, (int)d, signs.data_ptr<float>(),
                         boundaries.data_ptr<float>(), (int)bits, (int)codebook_class, kp.data_ptr<uint8_t>(),
                         reinterpret_cast<uint16_t*>(kn.data_ptr()), vp.data_ptr<uint8_t>(),
                         reinterpret_cast<uint16_t*>(vn.data_ptr()), stream_of(k)));
  return {kp, kn, vp, vn};
}

at::Tensor decode(const at::Tensor& packed, const at::Tensor& norms, const at::Tensor& levels, const at::Tensor& signs,
                  int64_t bits, int64_t d, c10::ScalarType out_dtype) {
  contig(packed, "packed");
  contig(norms, "norms");
  contig(levels, "levels");
  contig(signs, "signs");
  TORCH_CHECK(packed.scalar_type() == at::kByte && norms.scalar_type() == at::kHalf,
              "fused_tq: packed must be uint8 and norms float16");
  const c10::DeviceGuard g(packed.device());
  const int64_t n = norms.numel();
  auto sizes = norms.sizes().vec();
  sizes.push_back(d);
  at::Tensor out = at::empty(sizes, packed.options().dtype(out_dtype));
  check_rc(ftq_decode(packed.data_ptr<uint8_t>(), reinterpret_cast<const uint16_t*>(norms.data_ptr()), n, (int)d,
                      levels.data_ptr<float>(), signs.data_ptr<float>(), (int)bits, out.data_ptr(), dt_of(out_dtype),
                      stream_of(packed)));
  return out;
}

at::Tensor rht(const at::Tensor& x, const at::Tensor& signs, bool inverse, c10::ScalarType out_dtype) {
  contig(x, "x");
  contig(signs, "signs");
  const c10::DeviceGuard g(x.device());
  const int64_t d = x.size(-1);
  at::Tensor out = at::empty(x.sizes(), x.options().dtype(out_dtype));
  check_rc(ftq_rht(x.data_ptr(), dt(x), d > 0 ? x.numel() / d : 0, (int)d, signs.data_ptr<float>(), inverse ? 1 : 0,
                   out.data_ptr(), dt_of(out_dtype), stream_of(x)));
  return out;
}

// ---- paged library-format cache -----------------------------------------

void paged_store(const at::Tensor& key, const at::Tensor& value, at::Tensor& kv_cache, const at::Tensor& slot_mapping,
                 const at::Tensor& k_signs, const at::Tensor& v_signs, const at::Tensor& k_boundaries,
                 const at::Tensor& v_boundaries, int64_t bits_k, int64_t bits_v, int64_t page_size) {
  contig(key, "key");
  contig(value, "value");
  contig(kv_cache, "kv_cache");
  contig(slot_mapping, "slot_mapping");
  TORCH_CHECK(key.dim() == 3 && value.sizes() == key.sizes(), "fused_tq: key/value must be [n, Hkv, d]");
  TORCH_CHECK(key.scalar_type() == value.scalar_type(), "fused_tq: key and value dtypes differ");
  TORCH_CHECK(slot_mapping.scalar_type() == at::kLong, "fused_tq: slot_mapping must be int64");
  const c10::DeviceGuard g(key.device());
  check_rc(ftq_paged_store(key.data_ptr(), value.data_ptr(), dt(key), key.size(0), (int)key.size(1), (int)key.size(2),
                           k_signs.data_ptr<float>(), v_signs.data_ptr<float>(), k_boundaries.data_ptr<float>(),
                           v_boundaries.data_ptr<float>(), (int)bits_k, (int)bits_v, slot_mapping.data_ptr<int64_t>(),
                           kv_cache.data_ptr<uint8_t>(), (int)page_size, kv_cache.size(0), stream_of(key)));
}

void paged_decode_attention(const at::Tensor& query, const at::Tensor& kv_cache, const at::Tensor& block_table,
                            const at::Tensor& seq_lens, const at::Tensor& k_signs, const at::Tensor& v_signs,
                            const at::Tensor& k_levels, const at::Tensor& v_levels, int64_t bits_k, int64_t bits_v,
                            int64_t page_size, double scale, int64_t num_splits, at::Tensor& workspace,
                            at::Tensor& out, bool fp32_operands) {
  contig(query, "query");
  contig(kv_cache, "kv_cache");
  contig(block_table, "block_table");
  contig(seq_lens, "seq_lens");
  contig(workspace, "workspace");
  contig(out, "out");
  TORCH_CHECK(query.dim() == 3 && out.sizes() == query.sizes(), "fused_tq: query and out must be [B, Hq, d]");
  TORCH_CHECK(block_table.scalar_type() == at::kInt && seq_lens.scalar_type() == at::kInt,
              "fused_tq: block_table and seq_lens must be int32");
  const c10::DeviceGuard g(query.device());
  auto fn = fp32_operands ? ftq_paged_decode_attention_valu : ftq_paged_decode_attention;
  check_rc(fn(query.data_ptr(), dt(query), kv_cache.data_ptr<uint8_t>(), block_table.data_ptr<int32_t>(),
              seq_lens.data_ptr<int32_t>(), (int)query.size(0), (int)query.size(1), (int)kv_cache.size(1),
              (int)query.size(2), (int)page_size, (int)block_table.size(1), kv_cache.size(0),
              k_signs.data_ptr<float>(), v_signs.data_ptr<float>(), k_levels.data_ptr<float>(),
              v_levels.data_ptr<float>(), (int)bits_k, (int)bits_v, (float)scale, (int)num_splits,
              workspace.data_ptr(), workspace.numel() * workspace.element_size(), out.data_ptr(), dt(out),
              stream_of(query)));
}

// ---- vLLM v1 slot cache -------------------------------------------------

void v1_store(const at::Tensor& key, const at::Tensor& value, at::Tensor& kv_cache, const at::Tensor& slot_mapping,
              const at::Tensor& midpoints, int64_t key_bits, int64_t value_bits, int64_t v_flags,
              const std::optional<at::Tensor>& rotation, const std::optional<at::Tensor>& coeffs) {
  contig(key, "key");
  contig(value, "value");
  on_device(kv_cache, "kv_cache");
  contig(slot_mapping, "slot_mapping");
  contig(midpoints, "midpoints");
  TORCH_CHECK(key.dim() == 3 && value.sizes() == key.sizes(), "fused_tq: key/value must be [n, Hkv, d]");
  TORCH_CHECK(kv_cache.dim() == 4 && kv_cache.scalar_type() == at::kByte && kv_cache.stride(3) == 1,
              "fused_tq: kv_cache must be uint8 [num_blocks, block_size, Hkv, slot] with contiguous slots");
  TORCH_CHECK(slot_mapping.scalar_type() == at::kLong, "fused_tq: slot_mapping must be int64");
  const c10::DeviceGuard g(key.device());
  const int d = (int)key.size(2);
  if (coeffs.has_value()) {
    contig(*coeffs, "coeffs");
    check_rc(ftq_v1_store_blockdiag(key.data_ptr(), value.data_ptr(), dt(key), key.size(0), (int)key.size(1), d,
                                    midpoints.data_ptr<float>(), (int)key_bits, (int)value_bits, (int)v_flags,
                                    slot_mapping.data_ptr<int64_t>(), kv_cache.data_ptr<uint8_t>(), kv_cache.size(0),
                                    (int)kv_cache.size(1), kv_cache.stride(0), kv_cache.stride(1), kv_cache.stride(2),
                                    coeffs->data_ptr<float>(), (int)coeffs->size(0), stream_of(key)));
  } else {
    if (rotation.has_value()) contig(*rotation, "rotation");
    check_rc(ftq_v1_store_rot(key.data_ptr(), value.data_ptr(), dt(key), key.size(0), (int)key.size(1), d,
                              midpoints.data_ptr<float>(), (int)key_bits, (int)value_bits, (int)v_flags,
                              slot_mapping.data_ptr<int64_t>(), kv_cache.data_ptr<uint8_t>(), kv_cache.size(0),
                              (int)kv_cache.size(1), kv_cache.stride(0), kv_cache.stride(1), kv_cache.stride(2),
                              rotation.has_value() ? rotation->data_ptr<float>() : nullptr, stream_of(key)));
  }
}

void v1_decode_attention(const at::Tensor& query, const at::Tensor& kv_cache, const at::Tensor& block_table,
                         const at::Tensor& seq_lens, const std::optional<at::Tensor>& kv_start,
                         const at::Tensor& centroids, int64_t key_bits, int64_t value_bits, double scale,
                         int64_t v_flags, int64_t num_splits, at::Tensor& workspace, at::Tensor& out,
                         std::optional<at::Tensor> lse, const std::optional<at::Tensor>& rotation) {
  contig(query, "query");
  on_device(kv_cache, "kv_cache");
  contig(block_table, "block_table");
  contig(seq_lens, "seq_lens");
  contig(centroids, "centroids");
  contig(workspace, "workspace");
  contig(out, "out");
  TORCH_CHECK(query.dim() == 3 && out.sizes() == query.sizes(), "fused_tq: query and out must be [B, Hq, d]");
  TORCH_CHECK(kv_cache.dim() == 4 && kv_cache.scalar_type() == at::kByte && kv_cache.stride(3) == 1,
              "fused_tq: kv_cache must be uint8 [num_blocks, block_size, Hkv, slot] with contiguous slots");
  TORCH_CHECK(block_table.scalar_type() == at::kInt && seq_lens.scalar_type() == at::kInt,
              "fused_tq: block_table and seq_lens must be int32");
  if (kv_start.has_value()) contig(*kv_start, "kv_start");
  if (lse.has_value()) contig(*lse, "lse");
  if (rotation.has_value()) contig(*rotation, "rotation");
  const c10::DeviceGuard g(query.device());
  check_rc(ftq_v1_decode_attention_rot(
      query.data_ptr(), dt(query), kv_cache.data_ptr<uint8_t>(), kv_cache.size(0), (int)kv_cache.size(1),
      kv_cache.stride(0), kv_cache.stride(1), kv_cache.stride(2), block_table.data_ptr<int32_t>(),
      (int)block_table.size(1), seq_lens.data_ptr<int32_t>(),
      kv_start.has_value() ? kv_start->data_ptr<int32_t>() : nullptr, (int)query.size(0), (int)query.size(1),
      (int)kv_cache.size(2), (int)query.size(2), centroids.data_ptr<float>(), (int)key_bits, (int)value_bits,
      (float)scale, (int)v_flags, (int)num_splits, workspace.data_ptr(), workspace.numel() * workspace.element_size(),
      out.data_ptr(), dt(out), lse.has_value() ? lse->data_ptr<float>() : nullptr,
      rotation.has_value() ? rotation->data_ptr<float>() : nullptr, stream_of(query)));
}

// Causal attention of the last query.size(0) of past_len + query.size(0)
// stored positions of one sequence; the dequantised fragments and split
// partials live in a workspace from torch's caching allocator (as large as
// the chunk and its context need, returned to the stream's pool afterwards).
void v1_chunk_attention(const at::Tensor& query, const at::Tensor& kv_cache, const at::Tensor& block_row,
                        int64_t past_len, const std::optional<at::Tensor>& centroids, int64_t key_bits,
                        int64_t value_bits, double scale, int64_t v_flags, int64_t window, at::Tensor& out,
                        const std::optional<at::Tensor>& rotation) {
  contig(query, "query");
  on_device(kv_cache, "kv_cache");
  contig(block_row, "block_row");
  contig(out, "out");
  TORCH_CHECK(query.dim() == 3 && out.sizes() == query.sizes(), "fused_tq: query and out must be [n, Hq, d]");
  TORCH_CHECK(kv_cache.dim() == 4 && kv_cache.scalar_type() == at::kByte && kv_cache.stride(3) == 1,
              "fused_tq: kv_cache must be uint8 [num_blocks, block_size, Hkv, slot] with contiguous slots");
  TORCH_CHECK(block_row.scalar_type() == at::kInt, "fused_tq: block_row must be int32");
  TORCH_CHECK_VALUE(past_len >= 0 && past_len <= INT32_MAX && window >= 0 && window <= INT32_MAX &&
                        query.size(0) <= INT32_MAX && block_row.numel() <= INT32_MAX,
                    "fused_tq: past_len / window / token counts out of range");
  // the kernels read 2^key_bits centroids and a d x d rotation (raw slots and fp8 keys: no centroids)
  if (centroids.has_value()) {
    contig(*centroids, "centroids");
    TORCH_CHECK_VALUE(key_bits < 1 || key_bits > 8 || (v_flags & 4) != 0 || centroids->numel() == ((int64_t)1 << key_bits),
                      "fused_tq: centroids must have 2^key_bits entries");
  }
  if (rotation.has_value()) {
    contig(*rotation, "rotation");
    TORCH_CHECK_VALUE(rotation->numel() == query.size(2) * query.size(2), "fused_tq: rotation must be [d, d]");
  }
  const c10::DeviceGuard g(query.device());
  const int n = (int)query.size(0), hq = (int)query.size(1), d = (int)query.size(2), hkv = (int)kv_cache.size(2);
  if (n == 0) return;
  const int64_t need = ftq_v1_chunk_workspace_bytes(n, hq, hkv, d, (int)past_len, (int)key_bits, (int)value_bits,
                                                    (int)v_flags, (int)window);
  TORCH_CHECK_VALUE(need >= 0, "fused_tq: chunk attention does not take this head_dim, code width or token count");
  at::Tensor ws = at::empty({need}, query.options().dtype(at::kByte));
  check_rc(ftq_v1_chunk_attention(
      query.data_ptr(), dt(query), kv_cache.data_ptr<uint8_t>(), kv_cache.size(0), (int)kv_cache.size(1),
      kv_cache.stride(0), kv_cache.stride(1), kv_cache.stride(2), block_row.data_ptr<int32_t>(),
      (int)block_row.numel(), (int)past_len, n, hq, hkv, d,
      centroids.has_value() ? centroids->data_ptr<float>() : nullptr, (int)key_bits, (int)value_bits, (float)scale,
      (int)v_flags, (int)window, ws.data_ptr(), need, out.data_ptr(), dt(out),
      rotation.has_value() ? rotation->data_ptr<float>() : nullptr, stream_of(query)));
}

// ---- library-format attention: windows, other head dims, several tokens ----

void lib_attention(const at::Tensor& query_in, const at::Tensor& codes_k, const std::optional<at::Tensor>& codes_v,
                   const std::optional<at::Tensor>& norms_k, const std::optional<at::Tensor>& norms_v,
                   const std::optional<at::Tensor>& block_table, const at::Tensor& lens,
                   std::optional<at::Tensor> new_key, std::optional<at::Tensor> new_value,
                   const at::Tensor& k_signs, const at::Tensor& v_signs, const at::Tensor& k_levels,
                   const at::Tensor& v_levels, int64_t bits_k, int64_t bits_v, int64_t max_len, double scale,
                   int64_t window, int64_t sinks, bool precise, at::Tensor& out) {
  on_device(query_in, "query");
  on_device(out, "out");
  contig(codes_k, "codes_k");
  contig(lens, "lens");
  TORCH_CHECK(query_in.dim() == 4 && out.sizes() == query_in.sizes() && out.stride(3) == 1,
              "fused_tq: query and out must be [B, Hq, n, d], out with contiguous rows");
  const c10::DeviceGuard g(query_in.device());
  const at::Tensor query = rows16(query_in);
  TORCH_CHECK(lens.scalar_type() == at::kInt && lens.numel() == query.size(0), "fused_tq: lens must be int32 [B]");
  TORCH_CHECK(codes_k.scalar_type() == at::kByte && codes_k.dim() == 4, "fused_tq: codes_k must be uint8, 4-D");
  TORCH_CHECK_VALUE(max_len >= 0 && max_len <= INT32_MAX && window >= 0 && window <= INT32_MAX && sinks >= 0 &&
                        sinks <= INT32_MAX && query.size(2) <= INT32_MAX && query.size(0) <= INT32_MAX,
                    "fused_tq: max_len / window / sinks out of range");
  const bool paged = block_table.has_value();
  const int64_t B = query.size(0), d = query.size(3), hkv = codes_k.size(1);
  ftq_lib_attention_args a{};
  a.query = query.data_ptr();
  a.out = out.data_ptr();
  a.q_batch = query.stride(0); a.q_head = query.stride(1); a.q_row = query.stride(2);
  a.o_batch = out.stride(0); a.o_head = out.stride(1); a.o_row = out.stride(2);
  a.q_dtype = dt(query); a.out_dtype = dt(out);
  a.batch = (int)B; a.n_query = (int)query.size(2); a.num_q_heads = (int)query.size(1); a.num_kv_heads = (int)hkv;
  a.d = (int)d;
  a.paged = paged ? 1 : 0;
  a.codes_k = codes_k.data_ptr<uint8_t>();
  if (paged) {
    contig(*block_table, "block_table");
    TORCH_CHECK(block_table->scalar_type() == at::kInt && block_table->dim() == 2 && block_table->size(0) == B,
                "fused_tq: block_table must be int32 [B, max_blocks]");
    TORCH_CHECK(codes_k.size(3) == 2 * d * (bits_k + bits_v) + 64, "fused_tq: sub-block size does not match (d, bits)");
    a.block_table = block_table->data_ptr<int32_t>();
    a.page_size = (int)codes_k.size(2) * 16; a.max_blocks = (int)block_table->size(1); a.num_blocks = codes_k.size(0);
  } else {
    TORCH_CHECK(codes_v.has_value() && norms_k.has_value() && norms_v.has_value(), "fused_tq: flat codes and norms");
    contig(*codes_v, "codes_v");
    contig(*norms_k, "norms_k");
    contig(*norms_v, "norms_v");
    const int64_t cap = codes_k.size(2);
    TORCH_CHECK(codes_k.size(0) == B && codes_k.size(3) == d * bits_k / 8 && codes_v->scalar_type() == at::kByte &&
                    codes_v->dim() == 4 && codes_v->size(0) == B && codes_v->size(1) == hkv && codes_v->size(2) == cap &&
                    codes_v->size(3) == d * bits_v / 8,
                "fused_tq: flat codes must be [B, Hkv, capacity, d * bits / 8]");
    TORCH_CHECK(norms_k->scalar_type() == at::kHalf && norms_v->scalar_type() == at::kHalf &&
                    norms_k->numel() == B * hkv * cap && norms_v->numel() == B * hkv * cap,
                "fused_tq: flat norms must be float16 [B, Hkv, capacity]");
    a.codes_v = codes_v->data_ptr<uint8_t>();
    a.norms_k = reinterpret_cast<const uint16_t*>(norms_k->data_ptr());
    a.norms_v = reinterpret_cast<const uint16_t*>(norms_v->data_ptr());
    a.capacity = (int)cap;
  }
  a.lens = lens.data_ptr<int32_t>();
  a.max_len = (int)max_len;
  for (const at::Tensor* t : {&k_signs, &v_signs}) {
    contig(*t, "signs");
    TORCH_CHECK(t->numel() == d, "fused_tq: signs must have d entries");
  }
  contig(k_levels, "k_levels");
  contig(v_levels, "v_levels");
  TORCH_CHECK(bits_k >= 2 && bits_k <= 4 && bits_v >= 2 && bits_v <= 4 && k_levels.numel() == (1 << bits_k) &&
                  v_levels.numel() == (1 << bits_v),
              "fused_tq: levels must have 2^bits entries");
  a.k_signs = k_signs.data_ptr<float>(); a.v_signs = v_signs.data_ptr<float>();
  a.k_levels = k_levels.data_ptr<float>(); a.v_levels = v_levels.data_ptr<float>();
  a.bits_k = (int)bits_k; a.bits_v = (int)bits_v;
  if (new_key.has_value()) {
    TORCH_CHECK(new_value.has_value() && new_key->dim() == 4 && new_key->sizes() == new_value->sizes() &&
                    new_key->size(0) == B && new_key->size(1) == hkv && new_key->size(2) == query.size(2) &&
                    new_key->size(3) == d && new_key->scalar_type() == new_value->scalar_type(),
                "fused_tq: new keys and values must be [B, Hkv, n, d] of one type");
    on_device(*new_key, "new_key");
    on_device(*new_value, "new_value");
    new_key = rows16(*new_key);
    new_value = rows16(*new_value);
    a.new_key = new_key->data_ptr(); a.new_value = new_value->data_ptr(); a.new_dtype = dt(*new_key);
    a.k_batch = new_key->stride(0); a.k_head = new_key->stride(1); a.k_tok = new_key->stride(2);
    a.v_batch = new_value->stride(0); a.v_head = new_value->stride(1); a.v_tok = new_value->stride(2);
  }
  a.scale = (float)scale; a.window = (int)window; a.sinks = (int)sinks; a.precise = precise ? 1 : 0;
  if (B == 0 || query.size(2) == 0) return;
  const int64_t need = ftq_lib_attention_workspace_bytes(a.batch, a.n_query, a.num_q_heads, a.num_kv_heads, a.d,
                                                         a.max_len, a.window, a.sinks, a.precise, a.new_key == nullptr);
  TORCH_CHECK_VALUE(need >= 0, "fused_tq: library attention does not take these sizes");
  at::Tensor ws = at::empty({need}, query.options().dtype(at::kByte));
  check_rc(ftq_lib_attention(&a, ws.data_ptr(), need, stream_of(query)));
}

// ---- steps of the HuggingFace attention forward ----

// q [B, Hq, n, d], k [B, Hkv, n, d], cos / sin [B or 1, n, d]
// -> the embedded q and k, [B, H, n, d] views of [B, n, H, d] storage
std::tuple<at::Tensor, at::Tensor> rope(const at::Tensor& q_in, const at::Tensor& k_in, const at::Tensor& cos_in,
                                        const at::Tensor& sin_in) {
  on_device(q_in, "q");
  on_device(k_in, "k");
  on_device(cos_in, "cos");
  on_device(sin_in, "sin");
  const c10::DeviceGuard g(q_in.device());
  const at::Tensor q = rows16(q_in), k = rows16(k_in), cos = rows16(cos_in), sin = rows16(sin_in);
  TORCH_CHECK(q.dim() == 4 && k.dim() == 4 && q.size(0) == k.size(0) && q.size(2) == k.size(2) && q.size(3) == k.size(3),
              "fused_tq: q and k must be [B, H, n, d]");
  const int64_t B = q.size(0), n = q.size(2), d = q.size(3);
  for (const at::Tensor* t : {&cos, &sin})
    TORCH_CHECK(t->dim() == 3 && (t->size(0) == B || t->size(0) == 1) && t->size(1) == n && t->size(2) == d &&
                    t->scalar_type() == q.scalar_type(),
                "fused_tq: cos and sin must be [B or 1, n, d] of q's type");
  TORCH_CHECK(q.scalar_type() == k.scalar_type(), "fused_tq: q and k must be of one type");
  at::Tensor qo = at::empty({B, n, q.size(1), d}, q.options()), ko = at::empty({B, n, k.size(1), d}, k.options());
  if (qo.numel() > 0 && ko.numel() > 0)
    check_rc(ftq_rope(q.data_ptr(), qo.data_ptr(), q.stride(0), q.stride(1), q.stride(2), (int)q.size(1), k.data_ptr(),
                      ko.data_ptr(), k.stride(0), k.stride(1), k.stride(2), (int)k.size(1), cos.data_ptr(),
                      cos.size(0) == 1 ? 0 : cos.stride(0), cos.stride(1), sin.data_ptr(),
                      sin.size(0) == 1 ? 0 : sin.stride(0), sin.stride(1), dt(q), (int)B, (int)n, (int)d, stream_of(q)));
  return {qo.transpose(1, 2), ko.transpose(1, 2)};
}

at::Tensor append_slots(at::Tensor& lens, int64_t n, int64_t capacity) {
  contig(lens, "lens");
  TORCH_CHECK(lens.scalar_type() == at::kInt && n >= 0 && n <= INT32_MAX, "fused_tq: lens must be int32");
  const c10::DeviceGuard g(lens.device());
  at::Tensor slots = at::empty({lens.numel() * n}, lens.options().dtype(at::kLong));
  check_rc(ftq_append_slots(lens.data_ptr<int32_t>(), slots.data_ptr<int64_t>(), (int)lens.numel(), (int)n, capacity,
                            stream_of(lens)));
  return slots;
}

// ---- raw fp16 slots (boundary layers) -------------------------------------

void raw_store(const at::Tensor& key, const at::Tensor& value, at::Tensor& kv_cache, const at::Tensor& slot_mapping) {
  contig(key, "key");
  contig(value, "value");
  on_device(kv_cache, "kv_cache");
  contig(slot_mapping, "slot_mapping");
  TORCH_CHECK(key.dim() == 3 && value.sizes() == key.sizes(), "fused_tq: key/value must be [n, Hkv, d]");
  TORCH_CHECK(kv_cache.dim() == 4 && kv_cache.scalar_type() == at::kByte && kv_cache.stride(3) == 1,
              "fused_tq: kv_cache must be uint8 [num_blocks, block_size, Hkv, slot] with contiguous slots");
  const c10::DeviceGuard g(key.device());
  check_rc(ftq_raw_store(key.data_ptr(), value.data_ptr(), dt(key), key.size(0), (int)key.size(1), (int)key.size(2),
                         slot_mapping.data_ptr<int64_t>(), kv_cache.data_ptr<uint8_t>(), kv_cache.size(0),
                         (int)kv_cache.size(1), kv_cache.stride(0), kv_cache.stride(1), kv_cache.stride(2),
                         stream_of(key)));
}

void raw_decode_attention(const at::Tensor& query, const at::Tensor& kv_cache, const at::Tensor& block_table,
                          const at::Tensor& seq_lens, const std::optional<at::Tensor>& kv_start, double scale,
                          int64_t num_splits, at::Tensor& workspace, at::Tensor& out, std::optional<at::Tensor> lse) {
  contig(query, "query");
  on_device(kv_cache, "kv_cache");
  contig(block_table, "block_table");
  contig(seq_lens, "seq_lens");
  contig(workspace, "workspace");
  contig(out, "out");
  TORCH_CHECK(query.dim() == 3 && out.sizes() == query.sizes(), "fused_tq: query and out must be [B, Hq, d]");
  TORCH_CHECK(kv_cache.dim() == 4 && kv_cache.scalar_type() == at::kByte && kv_cache.stride(3) == 1,
              "fused_tq: kv_cache must be uint8 [num_blocks, block_size, Hkv, slot] with contiguous slots");
  if (kv_start.has_value()) contig(*kv_start, "kv_start");
  if (lse.has_value()) contig(*lse, "lse");
  const c10::DeviceGuard g(query.device());
  check_rc(ftq_raw_decode_attention_lse(
      query.data_ptr(), dt(query), kv_cache.data_ptr<uint8_t>(), kv_cache.size(0), (int)kv_cache.size(1),
      kv_cache.stride(0), kv_cache.stride(1), kv_cache.stride(2), block_table.data_ptr<int32_t>(),
      (int)block_table.size(1), seq_lens.data_ptr<int32_t>(),
      kv_start.has_value() ? kv_start->data_ptr<int32_t>() : nullptr, (int)query.size(0), (int)query.size(1),
      (int)kv_cache.size(2), (int)query.size(2), (float)scale, (int)num_splits, workspace.data_ptr(),
      workspace.numel() * workspace.element_size(), out.data_ptr(), dt(out),
      lse.has_value() ? lse->data_ptr<float>() : nullptr, stream_of(query)));
}

}  // namespace

TORCH_LIBRARY(fused_tq, m) {
  m.def("encode(Tensor x, Tensor signs, Tensor boundaries, int bits, int codebook_class) -> (Tensor, Tensor)");
  m.def("encode_kv(Tensor k, Tensor v, Tensor signs, Tensor boundaries, int bits, int codebook_class) -> "
        "(Tensor, Tensor, Tensor, Tensor)");
  m.def("decode(Tensor packed, Tensor norms, Tensor levels, Tensor signs, int bits, int d, ScalarType out_dtype) -> Tensor");
  m.def("rht(Tensor x, Tensor signs, bool inverse, ScalarType out_dtype) -> Tensor");
  m.def("paged_store(Tensor key, Tensor value, Tensor(a!) kv_cache, Tensor slot_mapping, Tensor k_signs, "
        "Tensor v_signs, Tensor k_boundaries, Tensor v_boundaries, int bits_k, int bits_v, int page_size) -> ()");
  m.def("paged_decode_attention(Tensor query, Tensor kv_cache, Tensor block_table, Tensor seq_lens, "
        "Tensor k_signs, Tensor v_signs, Tensor k_levels, Tensor v_levels, int bits_k, int bits_v, int page_size, "
        "float scale, int num_splits, Tensor(a!) workspace, Tensor(b!) out, bool fp32_operands) -> ()");
  m.def("v1_store(Tensor key, Tensor value, Tensor(a!) kv_cache, Tensor slot_mapping, Tensor midpoints, "
        "int key_bits, int value_bits, int v_flags, Tensor? rotation, Tensor? coeffs) -> ()");
  m.def("v1_decode_attention(Tensor query, Tensor kv_cache, Tensor block_table, Tensor seq_lens, "
        "Tensor? kv_start, Tensor centroids, int key_bits, int value_bits, float scale, int v_flags, "
        "int num_splits, Tensor(a!) workspace, Tensor(b!) out, Tensor(c!)? lse, Tensor? rotation) -> ()");
  m.def("v1_chunk_attention(Tensor query, Tensor kv_cache, Tensor block_row, int past_len, Tensor? centroids, "
        "int key_bits, int value_bits, float scale, int v_flags, int window, Tensor(a!) out, Tensor? rotation) -> ()");
  m.def("lib_attention(Tensor query, Tensor codes_k, Tensor? codes_v, Tensor? norms_k, Tensor? norms_v, "
        "Tensor? block_table, Tensor lens, Tensor? new_key, Tensor? new_value, Tensor k_signs, Tensor v_signs, "
        "Tensor k_levels, Tensor v_levels, int bits_k, int bits_v, int max_len, float scale, int window, int sinks, "
        "bool precise, Tensor(a!) out) -> ()");
  m.def("rope(Tensor q, Tensor k, Tensor cos, Tensor sin) -> (Tensor, Tensor)");
  m.def("append_slots(Tensor(a!) lens, int n, int capacity) -> Tensor");
  m.def("raw_store(Tensor key, Tensor value, Tensor(a!) kv_cache, Tensor slot_mapping) -> ()");
  m.def("raw_decode_attention(Tensor query, Tensor kv_cache, Tensor block_table, Tensor seq_lens, "
        "Tensor? kv_start, float scale, int num_splits, Tensor(a!) workspace, Tensor(b!) out, "
        "Tensor(c!)? lse) -> ()");
}

TORCH_LIBRARY_IMPL(fused_tq, CUDA, m) {
  m.impl("encode", &encode);
  m.impl("encode_kv", &encode_kv);
  m.impl("decode", &decode);
  m.impl("rht", &rht);
  m.impl("paged_store", &paged_store);
  m.impl("paged_decode_attention", &paged_decode_attention);
  m.impl("v1_store", &v1_store);
  m.impl("v1_decode_attention", &v1_decode_attention);
  m.impl("v1_chunk_attention", &v1_chunk_attention);
  m.impl("lib_attention", &lib_attention);
  m.impl("rope", &rope);
  m.impl("append_slots", &append_slots);
  m.impl("raw_store", &raw_store);
  m.impl("raw_decode_attention", &raw_decode_attention);
}
