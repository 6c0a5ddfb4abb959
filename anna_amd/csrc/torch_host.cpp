// Host side of the calls a decode step repeats, on torch's C++ tensors: the checks, the output and
// workspace allocations and the argument blocks of anna_mi.h, which took 15 to 60 us a call in Python
// (linear 17 us around a 3.7 us kernel, a packed-cache decode 35 us, the sparse block 65 us).
//
// Every function here takes only the plain case of its Python caller -- tensors of the right types,
// shapes, layouts and device -- and answers None to anything else, without side effects; the caller
// then goes its general way, which converts or refuses as it always did.  Nothing is kept between
// calls: each one reads the tensors it is given.
//
// The library is not linked: Python hands over the addresses of its entry points (bind), so that its
// stamp check and its error text stay in one place.  The stream is an argument (the caller's current
// stream), so no device header is needed.
#include <pybind11/pybind11.h>
#include <torch/csrc/utils/pybind.h>

#include <ATen/ATen.h>
#include <ATen/core/grad_mode.h>

#include <cstdlib>
#include <optional>
#include <stdexcept>
#include <string>

#include "../../include/anna_mi.h"

namespace py = pybind11;
using at::Tensor;
using OptTensor = std::optional<Tensor>;

namespace {

struct Library {
  decltype(&anna_mi_last_error) last_error = nullptr;
  decltype(&anna_mi_int4_linear) int4_linear = nullptr;
  decltype(&anna_mi_decode_num_blocks) decode_num_blocks = nullptr;
  decltype(&anna_mi_gqa_decode_splitkv) gqa_decode_splitkv = nullptr;
  decltype(&anna_mi_tq_decode) tq_decode = nullptr;
  decltype(&anna_mi_tq_store) tq_store = nullptr;
  decltype(&anna_mi_moe_route_small) moe_route_small = nullptr;
  decltype(&anna_mi_moe_gather) moe_gather = nullptr;
  decltype(&anna_mi_moe_router) moe_router = nullptr;
  decltype(&anna_mi_moe_dispatch) moe_dispatch = nullptr;
  decltype(&anna_mi_moe_grouped_int4_mlp) moe_grouped_int4_mlp = nullptr;
  decltype(&anna_mi_moe_combine) moe_combine = nullptr;
  decltype(&anna_mi_moe_prefill_workspace) moe_prefill_workspace = nullptr;
  decltype(&anna_mi_moe_prefill) moe_prefill = nullptr;
} lib;

void bind(const py::dict& d) {
  auto get = [&](const char* name, auto& fn) {
    fn = reinterpret_cast<std::decay_t<decltype(fn)>>(d[name].cast<uintptr_t>());
  };
  get("anna_mi_last_error", lib.last_error);
  get("anna_mi_int4_linear", lib.int4_linear);
  get("anna_mi_decode_num_blocks", lib.decode_num_blocks);
  get("anna_mi_gqa_decode_splitkv", lib.gqa_decode_splitkv);
  get("anna_mi_tq_decode", lib.tq_decode);
  get("anna_mi_tq_store", lib.tq_store);
  get("anna_mi_moe_route_small", lib.moe_route_small);
  get("anna_mi_moe_gather", lib.moe_gather);
  get("anna_mi_moe_router", lib.moe_router);
  get("anna_mi_moe_dispatch", lib.moe_dispatch);
  get("anna_mi_moe_grouped_int4_mlp", lib.moe_grouped_int4_mlp);
  get("anna_mi_moe_combine", lib.moe_combine);
  get("anna_mi_moe_prefill_workspace", lib.moe_prefill_workspace);
  get("anna_mi_moe_prefill", lib.moe_prefill);
}

void check(int rc, const char* name) {
  if (rc != 0)
    throw std::runtime_error(std::string(name) + " failed (" + std::to_string(rc) + "): " + lib.last_error());
}

int dtype_code(const Tensor& t) {
  switch (t.scalar_type()) {
    case at::kBFloat16: return ANNA_MI_BF16;
    case at::kHalf: return ANNA_MI_F16;
    case at::kFloat: return ANNA_MI_F32;
    default: return -1;
  }
}

// A plain strided tensor with memory of its own on `dev` (not a fake, batched or sparse one)
bool plain(const Tensor& t, const at::Device& dev) {
  return t.defined() && t.layout() == at::kStrided && t.device() == dev && t.has_storage() &&
         t.unsafeGetTensorImpl()->key_set().has(c10::DispatchKey::CUDA) &&
         !t.unsafeGetTensorImpl()->key_set().has(c10::DispatchKey::Python) && !t.is_conj() && !t.is_neg();
}
bool plain(const OptTensor& t, const at::Device& dev) { return !t || plain(*t, dev); }
bool is(const Tensor& t, const at::Device& dev, at::ScalarType dt) {
  return plain(t, dev) && t.scalar_type() == dt && t.is_contiguous();
}

void* ptr(const Tensor& t) { return t.data_ptr(); }
void* ptr(const OptTensor& t) { return t ? t->data_ptr() : nullptr; }
void* stream_ptr(uintptr_t s) { return reinterpret_cast<void*>(s); }

// ---------------------------------------------------------------- int4 linear

// y = x . dequant(W)^T + bias for x [..., K] of the activation dtype (the tensors and conditions of
// fused_ops._check_int4_inputs).  `compute`: the layer's dtype.
OptTensor int4_linear(const Tensor& x, const Tensor& qw, const Tensor& qs, const Tensor& qz, const OptTensor& bias,
                      int64_t group, int64_t out_features, at::ScalarType compute, uintptr_t stream, bool strategies) {
  // a strategy other than the kernels' is the general path's to read
  if (const char* s = strategies ? std::getenv("ANNA_XPU_INT4_MATMUL") : nullptr; s && *s) return std::nullopt;
  const at::Device dev = x.device();
  if (!dev.is_cuda() || !plain(x, dev) || x.dim() < 1 || x.scalar_type() != compute || dtype_code(x) < 0 || x.numel() == 0)
    return std::nullopt;
  if (!is(qw, dev, at::kInt) || !plain(qs, dev) || dtype_code(qs) < 0 || !qs.is_contiguous() || !is(qz, dev, at::kChar))
    return std::nullopt;
  const int64_t K = x.size(-1), rows = x.numel() / K;
  if (qw.dim() != 2 || qs.dim() != 2 || qz.dim() != 2 || group <= 0 || qw.size(0) != out_features ||
      qw.size(1) * 8 < K || qs.size(1) != qw.size(0) || qz.sizes() != qs.sizes() || qs.size(0) * group < K)
    return std::nullopt;
  if (bias && (!plain(bias, dev) || (bias->requires_grad() && at::GradMode::is_enabled()) || bias->scalar_type() != compute || bias->dim() != 1 || bias->size(0) != out_features))
    return std::nullopt;
  int64_t row_stride = K;
  if (x.dim() == 2) {
    if (x.stride(1) != 1 || (rows > 1 && x.stride(0) < K)) return std::nullopt;
    if (rows > 1) row_stride = x.stride(0);
  } else if (!x.is_contiguous()) {
    return std::nullopt;
  }
  at::DimVector shape(x.sizes().begin(), x.sizes().end());
  shape.back() = out_features;
  Tensor y = at::empty(shape, x.options().requires_grad(false));
  check(lib.int4_linear(ptr(x), dtype_code(x), rows, K, row_stride, (const int32_t*)ptr(qw), out_features, qw.size(1),
                        ptr(qs), dtype_code(qs), (const int8_t*)ptr(qz), qs.size(0), group, ptr(y), stream_ptr(stream)),
        "anna_mi_int4_linear");
  if (bias) y.add_(bias->detach());
  return y;
}

// ---------------------------------------------------------------- split-KV decode with per-row lengths

anna_mi_view view(const Tensor& t, bool heads_only = false) {
  anna_mi_view v{ptr(t), t.stride(0), t.stride(1), t.stride(2), 0};
  if (!heads_only) v.s3 = t.stride(3);
  return v;
}
// [B, Hq, D] or [B, Hq, 1, D] as [B, Hq, 1, D]
anna_mi_view query_view(const Tensor& t) {
  return t.dim() == 3 ? anna_mi_view{ptr(t), t.stride(0), t.stride(1), 0, t.stride(2)} : view(t);
}

// One decode over [quantized slots ++ window] of every row: keys dense in the query's dtype or TQ-MSE
// codes (key_norms given), values in min/max groups.  query, gate, out: [B, Hq, D] or [B, Hq, 1, D].
// Without partial buffers they are allocated here; None also where given ones hold too few blocks.
OptTensor decode_rows(const Tensor& q, const OptTensor& gate, const OptTensor& out_in, const OptTensor& key,
                      const OptTensor& key_norms, const OptTensor& vdata, const OptTensor& vscales,
                      const OptTensor& vzeros, const Tensor& rk, const Tensor& rv, const Tensor& seq_lengths,
                      const Tensor& rotation, const Tensor& rotation_t, const Tensor& centroids, const OptTensor& signs,
                      const OptTensor& query_rot, const OptTensor& partial_stats, const OptTensor& partial_values,
                      int64_t bits, int64_t value_group, double scaling, int64_t block_size, bool tq_keys, uintptr_t stream) {
  const at::Device dev = q.device();
  const int dt = dtype_code(q);
  if (!dev.is_cuda() || dt < 0 || !plain(q, dev) || (q.dim() != 3 && q.dim() != 4)) return std::nullopt;
  for (const Tensor* t : {&rk, &rv, &seq_lengths, &rotation, &rotation_t, &centroids})
    if (!plain(*t, dev)) return std::nullopt;
  for (const OptTensor* t : {&gate, &out_in, &key, &key_norms, &vdata, &vscales, &vzeros, &signs, &query_rot,
                             &partial_stats, &partial_values})
    if (!plain(*t, dev)) return std::nullopt;
  const int64_t B = q.size(0), hq = q.size(1), D = q.size(-1);
  if (q.dim() == 4 && q.size(2) != 1) return std::nullopt;
  if (gate && (gate->sizes() != q.sizes() || gate->scalar_type() != q.scalar_type())) return std::nullopt;
  if (rk.dim() != 4 || rv.dim() != 4 || rk.size(0) != B || rk.size(3) != D || rv.sizes() != rk.sizes() ||
      rk.scalar_type() != q.scalar_type() || rv.scalar_type() != q.scalar_type())
    return std::nullopt;
  const int64_t H = rk.size(1);
  if (H < 1 || hq % H != 0 || value_group <= 0 || D % value_group != 0) return std::nullopt;
  if (seq_lengths.scalar_type() != at::kInt || seq_lengths.numel() != B || !seq_lengths.is_contiguous()) return std::nullopt;
  const int64_t per = bits == 2 ? 4 : 2;
  const int64_t C = vdata ? vdata->size(2) : 0;
  if (C > 0) {
    if (!key || !vscales || !vzeros || (tq_keys && !key_norms)) return std::nullopt;
    auto rows = [&](const Tensor& t, int64_t last) {
      return t.dim() == 4 && t.size(0) == B && t.size(1) == H && t.size(2) == C && t.size(3) == last;
    };
    if (!rows(*vdata, D / per) || vdata->scalar_type() != at::kByte || !rows(*vscales, D / value_group) ||
        !rows(*vzeros, D / value_group) || vscales->scalar_type() != q.scalar_type() ||
        vzeros->scalar_type() != q.scalar_type())
      return std::nullopt;
    if (tq_keys ? (!rows(*key, D / per) || key->scalar_type() != at::kByte || key_norms->scalar_type() != at::kHalf ||
                   key_norms->dim() != 3 || key_norms->size(0) != B || key_norms->size(1) != H || key_norms->size(2) != C)
                : (!rows(*key, D) || key->scalar_type() != q.scalar_type()))
      return std::nullopt;
  }
  const bool own = !query_rot;
  if (own != !partial_stats || own != !partial_values) return std::nullopt;
  if (!own && (partial_stats->scalar_type() != at::kFloat || partial_values->scalar_type() != at::kFloat ||
               query_rot->scalar_type() != at::kFloat || query_rot->numel() < B * hq * D || !query_rot->is_contiguous() ||
               partial_stats->dim() != 4 || partial_values->dim() != 4 || partial_stats->size(0) != B ||
               partial_stats->size(1) != hq || partial_values->size(0) != B || partial_values->size(1) != hq ||
               partial_values->size(3) != D))
    return std::nullopt;
  if (signs && (signs->scalar_type() != at::kFloat || signs->numel() != D)) return std::nullopt;
  if (out_in && (out_in->sizes() != q.sizes() || out_in->scalar_type() != q.scalar_type())) return std::nullopt;

  anna_mi_decode_args a{};
  a.dtype = dt;
  a.batch = B, a.q_heads = hq, a.kv_heads = H, a.head_dim = D;
  a.query = query_view(q);
  a.len1 = C;
  a.key_format = tq_keys ? 1 : 0;
  a.value_format = 1;
  if (C > 0) {
    a.key = view(*key);
    if (tq_keys) a.key_norms = view(*key_norms, true);
    a.value = view(*vdata);
    a.value_scales = view(*vscales);
    a.value_zeros = view(*vzeros);
  }
  a.key_bits = a.value_bits = (int)bits;
  a.value_group_size = value_group;
  a.rotation = (const float*)ptr(rotation);
  a.rotation_t = (const float*)ptr(rotation_t);
  a.key_centroids = (const float*)ptr(centroids);
  a.rotation_signs = (const float*)ptr(signs);
  a.len2 = rk.size(2);
  a.residual_key = view(rk);
  a.residual_value = view(rv);
  a.scaling = (float)scaling;
  a.block_size = block_size;
  a.seq_lengths = (const int32_t*)ptr(seq_lengths);
  const int64_t nblk = lib.decode_num_blocks(&a);
  Tensor ws;
  if (own) {
    ws = at::empty({B * hq * (D + nblk * (2 + D))}, q.options().dtype(at::kFloat).requires_grad(false));
    float* const w0 = (float*)ptr(ws);
    a.query_rot = w0;
    a.partial_values = {w0 + B * hq * D, hq * nblk * D, nblk * D, D, 1};
    a.partial_stats = {w0 + B * hq * D * (1 + nblk), hq * nblk * 2, nblk * 2, 2, 1};
    a.partial_capacity = nblk;
  } else {
    a.query_rot = (float*)ptr(query_rot);
    a.partial_stats = view(*partial_stats);
    a.partial_values = view(*partial_values);
    a.partial_capacity = std::min(partial_stats->size(2), partial_values->size(2));
    if (nblk > a.partial_capacity) return std::nullopt;
  }
  Tensor out = out_in ? *out_in : at::empty(q.sizes(), q.options().requires_grad(false));
  a.out = query_view(out);
  if (gate) {
    a.gate_layout = 2;
    a.gate = query_view(*gate);
  }
  check(lib.gqa_decode_splitkv(&a, stream_ptr(stream)), "anna_mi_gqa_decode_splitkv");
  return out;
}

// ---------------------------------------------------------------- 2-bit pool decode

// TurboQuantBatchCache.decode: contiguous bf16 [B, Hq, 256] query (and gate), the cache's own buffers.
OptTensor decode_pool(const Tensor& q, const OptTensor& gate, const OptTensor& out_in, const Tensor& key_codes,
                      const Tensor& key_norms, const Tensor& value_codes, const Tensor& value_norms, const Tensor& rk,
                      const Tensor& rvt, const Tensor& seq_offsets, const Tensor& seq_lengths, const Tensor& signs,
                      const Tensor& partial_stats, const Tensor& partial_values, const Tensor& item_table,
                      int64_t pool_tokens, int64_t window, int64_t kv_heads, int64_t q_heads, int64_t batch,
                      int64_t blocks_per_item, int64_t num_workgroups, double key_scale, double value_scale,
                      double scaling, uintptr_t stream) {
  const at::Device dev = key_codes.device();
  if (!dev.is_cuda() || !is(q, dev, at::kBFloat16) || q.dim() != 3 || q.size(0) != batch || q.size(1) != q_heads ||
      q.size(2) != 256)
    return std::nullopt;
  if (gate && (!is(*gate, dev, at::kBFloat16) || gate->sizes() != q.sizes())) return std::nullopt;
  if (out_in && (!is(*out_in, dev, at::kBFloat16) || out_in->sizes() != q.sizes())) return std::nullopt;
  for (const Tensor* t : {&key_codes, &key_norms, &value_codes, &value_norms, &rk, &rvt, &seq_offsets, &seq_lengths, &signs,
                          &partial_stats, &partial_values, &item_table})
    if (!plain(*t, dev) || !t->is_contiguous()) return std::nullopt;
  Tensor out = out_in ? *out_in : at::empty(q.sizes(), q.options().requires_grad(false));
  anna_mi_tq_decode_args a{};
  a.batch = batch, a.q_heads = q_heads, a.kv_heads = kv_heads, a.head_dim = 256;
  a.key_bits = a.value_bits = 2;
  a.query = (const uint16_t*)ptr(q);
  a.gate = (const uint16_t*)ptr(gate);
  a.key_codes = (const uint8_t*)ptr(key_codes);
  a.key_norms = (const uint16_t*)ptr(key_norms);
  a.value_codes = (const uint8_t*)ptr(value_codes);
  a.value_norms = (const uint16_t*)ptr(value_norms);
  a.pool_tokens = pool_tokens;
  a.residual_key = (const uint16_t*)ptr(rk);
  a.residual_value_t = (const uint16_t*)ptr(rvt);
  a.residual_capacity = window;
  a.seq_offsets = (const int32_t*)ptr(seq_offsets);
  a.seq_lengths = (const int32_t*)ptr(seq_lengths);
  a.signs = (const float*)ptr(signs);
  a.key_scale = (float)key_scale, a.value_scale = (float)value_scale, a.scaling = (float)scaling;
  a.blocks_per_item = blocks_per_item;
  a.num_workgroups = num_workgroups;
  a.partial_stats = (float*)ptr(partial_stats);
  a.partial_values = (float*)ptr(partial_values);
  a.item_table = (int32_t*)ptr(item_table);
  a.out = (uint16_t*)ptr(out);
  check(lib.tq_decode(&a, stream_ptr(stream)), "anna_mi_tq_decode");
  return out;
}

// ---------------------------------------------------------------- one-launch append

// anna_mi_tq_store into slab tensors of one layer; key_signs etc. only for inner-product keys.  Returns
// the lengths before (int64 [batch]).
OptTensor tq_store(const Tensor& k, const Tensor& v, const OptTensor& key_codes, const OptTensor& key_norms,
                   const OptTensor& key_signs, const OptTensor& key_residual_norms, const OptTensor& key_dense,
                   const OptTensor& vdata, const OptTensor& vscales, const OptTensor& vzeros, const Tensor& rk,
                   const Tensor& rv, const Tensor& seq_in, const Tensor& seq_out, const Tensor& seq_lengths,
                   const Tensor& signs,
                   const Tensor& thresholds, const OptTensor& centroids, const OptTensor& gaussian,
                   const OptTensor& gaussian_t, bool ip, int64_t row0, int64_t capacity, int64_t bits,
                   int64_t value_group, int64_t max_leaving, int64_t max_fill, uintptr_t stream) {
  const at::Device dev = rk.device();
  const int dt = dtype_code(rk);
  if (!dev.is_cuda() || dt < 0) return std::nullopt;
  const int64_t per = 16 / (int64_t)rk.element_size();
  for (const Tensor* t : {&k, &v}) {
    if (!plain(*t, dev) || t->dim() != 4 || t->scalar_type() != rk.scalar_type() || t->stride(3) != 1 ||
        t->stride(0) % per || t->stride(1) % per || t->stride(2) % per || (uintptr_t)ptr(*t) % 16 || t->size(2) == 0)
      return std::nullopt;
  }
  if (k.sizes() != v.sizes() || rk.dim() != 4 || k.size(1) != rk.size(1) || k.size(3) != rk.size(3) ||
      row0 < 0 || row0 + k.size(0) > rk.size(0) || !plain(rk, dev) || !plain(rv, dev) || !rk.is_contiguous() ||
      !rv.is_contiguous())
    return std::nullopt;
  for (const Tensor* t : {&seq_in, &seq_out, &seq_lengths, &signs, &thresholds})
    if (!plain(*t, dev) || !t->is_contiguous()) return std::nullopt;
  for (const OptTensor* t : {&key_codes, &key_norms, &key_signs, &key_residual_norms, &key_dense, &vdata, &vscales, &vzeros,
                             &centroids, &gaussian, &gaussian_t})
    if (*t && (!plain(**t, dev) || !(*t)->is_contiguous())) return std::nullopt;
  const int64_t batch = rk.size(0);
  Tensor past = at::empty({batch}, k.options().dtype(at::kLong).requires_grad(false));
  anna_mi_tq_store_args a{};
  a.dtype = dt, a.key_format = ip ? 1 : 0;
  a.batch = batch, a.row0 = row0, a.rows = k.size(0);
  a.kv_heads = k.size(1), a.head_dim = k.size(3), a.tokens = k.size(2);
  a.capacity = capacity, a.residual_capacity = rk.size(2);
  a.key_bits = a.value_bits = (int)bits;
  a.value_group_size = value_group;
  a.new_key = ptr(k), a.new_value = ptr(v);
  a.key_stride_row = k.stride(0), a.key_stride_head = k.stride(1), a.key_stride_token = k.stride(2);
  a.value_stride_row = v.stride(0), a.value_stride_head = v.stride(1), a.value_stride_token = v.stride(2);
  a.key_codes = (uint8_t*)ptr(key_codes);
  a.key_norms = ptr(key_norms);
  a.key_signs = (uint8_t*)ptr(key_signs);
  a.key_residual_norms = (float*)ptr(key_residual_norms);
  a.key_dense = ptr(key_dense);
  a.value_data = (uint8_t*)ptr(vdata);
  a.value_scales = ptr(vscales);
  a.value_zeros = ptr(vzeros);
  a.residual_key = ptr(rk), a.residual_value = ptr(rv);
  a.seq_in = (const int32_t*)ptr(seq_in);
  a.seq_out = (int32_t*)ptr(seq_out);
  a.seq_lengths = (int32_t*)ptr(seq_lengths);
  a.past_out = (int64_t*)ptr(past);
  a.max_leaving = max_leaving, a.max_fill = max_fill;
  a.signs = (const float*)ptr(signs);
  a.thresholds = (const float*)ptr(thresholds);
  a.centroids = (const float*)ptr(centroids);
  a.gaussian = (const float*)ptr(gaussian);
  a.gaussian_t = (const float*)ptr(gaussian_t);
  check(lib.tq_store(&a, stream_ptr(stream)), "anna_mi_tq_store");
  return past;
}

// ---------------------------------------------------------------- sparse MoE block

// Pieces of one workspace tensor, 256-byte aligned
struct Carve {
  size_t used = 0;
  size_t take(size_t bytes) {
    const size_t at = used;
    used += (bytes + 255) & ~size_t(255);
    return at;
  }
};

// The launches of SparseMoeInt4.forward (see anna_amd/moe.py) over one workspace allocation.
OptTensor moe_block(const Tensor& x, const Tensor& logits, const Tensor& gq, const Tensor& gs, const Tensor& gz,
                    const Tensor& uq, const Tensor& us, const Tensor& uz, const Tensor& dq, const Tensor& ds,
                    const Tensor& dz, const Tensor& experts, const Tensor& slots, int64_t group, int64_t top_k,
                    bool normalize, bool small, int64_t max_routes_hint, uintptr_t stream) {
  const at::Device dev = x.device();
  if (!dev.is_cuda() || !plain(x, dev) || !plain(logits, dev) || x.dim() != 2 || logits.dim() != 2) return std::nullopt;
  const int dt = dtype_code(x), ldt = dtype_code(logits), sdt = dtype_code(gs);
  if (dt < 0 || ldt < 0 || sdt < 0 || x.stride(1) != 1 || logits.stride(1) != 1) return std::nullopt;
  const int64_t T = x.size(0), H = x.size(1), E = logits.size(1), R = T * top_k;
  if (T < 1 || logits.size(0) != T || top_k < 1 || top_k > E || x.stride(0) < H || logits.stride(0) < E) return std::nullopt;
  for (const Tensor* t : {&gq, &uq, &dq})
    if (!is(*t, dev, at::kInt) || t->dim() != 3) return std::nullopt;
  for (const Tensor* t : {&gz, &uz, &dz})
    if (!is(*t, dev, at::kChar) || t->dim() != 3) return std::nullopt;
  for (const Tensor* t : {&gs, &us, &ds})
    if (!is(*t, dev, gs.scalar_type()) || t->dim() != 3) return std::nullopt;
  if (gq.sizes() != uq.sizes() || gs.sizes() != us.sizes()) return std::nullopt;
  if (!is(experts, dev, at::kLong) || !is(slots, dev, at::kLong) || experts.numel() != E || slots.numel() != E)
    return std::nullopt;
  const int64_t I = gq.size(1);
  if (dq.size(1) == H && ds.size(2) == H && gs.size(2) == I) {
    anna_mi_moe_prefill_args p{};
    p.dtype = dt, p.logits_dtype = ldt, p.scale_dtype = sdt, p.normalize = normalize;
    p.tokens = T, p.num_experts = E, p.top_k = top_k, p.hidden_dim = H, p.intermediate_dim = I, p.group_size = group;
    p.hidden = ptr(x), p.hidden_row_stride = T > 1 ? x.stride(0) : std::max(H, x.stride(0));
    p.logits = ptr(logits), p.logits_row_stride = logits.stride(0);
    p.slots = (const int64_t*)ptr(slots);
    p.gate_qweight = (const int32_t*)ptr(gq), p.gate_qscale = ptr(gs), p.gate_qzeros = (const int8_t*)ptr(gz);
    p.up_qweight = (const int32_t*)ptr(uq), p.up_qscale = ptr(us), p.up_qzeros = (const int8_t*)ptr(uz);
    p.down_qweight = (const int32_t*)ptr(dq), p.down_qscale = ptr(ds), p.down_qzeros = (const int8_t*)ptr(dz);
    p.hidden_packed_cols = gq.size(2), p.hidden_groups = gs.size(1);
    p.intermediate_packed_cols = dq.size(2), p.intermediate_groups = ds.size(1);
    if (const int64_t bytes = lib.moe_prefill_workspace(&p); bytes > 0) {
      Tensor ws = at::empty({bytes}, x.options().dtype(at::kByte).requires_grad(false));
      Tensor out = at::empty({T, H}, x.options().requires_grad(false));
      p.workspace = ptr(ws), p.out = ptr(out);
      check(lib.moe_prefill(&p, stream_ptr(stream)), "anna_mi_moe_prefill");
      return out;
    }
  }
  const size_t es = (size_t)x.element_size();
  Carve c;
  const size_t o_w = c.take(R * 4), o_sel = c.take(R * 8), o_usage = c.take(E * 4), o_off = c.take((E + 1) * 8),
               o_tok = c.take(R * 8), o_route = c.take(R * 8), o_pos = c.take(R * 8), o_items = c.take((4 + 4 * E) * 4),
               o_cw = c.take(R * es), o_x = c.take(R * H * es), o_y = c.take(R * H * es), o_act = c.take(R * I * 4);
  Tensor ws = at::empty({(int64_t)c.used}, x.options().dtype(at::kByte).requires_grad(false));
  Tensor out = at::empty({T, H}, x.options().requires_grad(false));
  char* const w0 = (char*)ptr(ws);
  float* const w = (float*)(w0 + o_w);
  int64_t *const sel = (int64_t*)(w0 + o_sel), *const off = (int64_t*)(w0 + o_off), *const tok = (int64_t*)(w0 + o_tok),
                 *const route = (int64_t*)(w0 + o_route), *const pos = (int64_t*)(w0 + o_pos);
  int32_t *const usage = (int32_t*)(w0 + o_usage), *const items = (int32_t*)(w0 + o_items);
  void* const st = stream_ptr(stream);
  if (small) {
    check(lib.moe_route_small(ptr(logits), ldt, T, E, logits.stride(0), top_k, normalize, w, sel, usage, off, tok, route, pos,
                              (const int64_t*)ptr(slots), items, st),
          "anna_mi_moe_route_small");
    check(lib.moe_gather(ptr(x), dt, H, x.stride(0), w, ANNA_MI_F32, route, R, top_k, w0 + o_x, w0 + o_cw, st),
          "anna_mi_moe_gather");
  } else {
    check(lib.moe_router(ptr(logits), ldt, T, E, logits.stride(0), top_k, normalize, w, sel, usage, st),
          "anna_mi_moe_router");
    check(lib.moe_dispatch(ptr(x), dt, T, H, x.stride(0), w, ANNA_MI_F32, sel, usage, 0, E, top_k, tok, route, off, w0 + o_x,
                           w0 + o_cw, pos, (const int64_t*)ptr(slots), items, st),
          "anna_mi_moe_dispatch");
  }
  anna_mi_moe_mlp_args a{};
  a.dtype = dt, a.scale_dtype = sdt;
  a.routes = R, a.hidden_dim = H, a.intermediate_dim = I;
  a.compact_hidden = w0 + o_x, a.compact_weights = w0 + o_cw, a.compact_outputs = w0 + o_y;
  a.expert_offsets = off;
  a.active_experts = (const int64_t*)ptr(experts), a.active_slots = (const int64_t*)ptr(slots), a.active_count = E;
  a.gate_qweight = (const int32_t*)ptr(gq), a.gate_qscale = ptr(gs), a.gate_qzeros = (const int8_t*)ptr(gz);
  a.up_qweight = (const int32_t*)ptr(uq), a.up_qscale = ptr(us), a.up_qzeros = (const int8_t*)ptr(uz);
  a.down_qweight = (const int32_t*)ptr(dq), a.down_qscale = ptr(ds), a.down_qzeros = (const int8_t*)ptr(dz);
  a.hidden_packed_cols = gq.size(2), a.hidden_groups = gs.size(1);
  a.intermediate_packed_cols = dq.size(2), a.intermediate_groups = ds.size(1);
  a.group_size = group;
  a.activation = (float*)(w0 + o_act);
  a.sweep_chunks = (int)std::min<int64_t>(4, std::max<int64_t>(1, (max_routes_hint + 15) / 16));
  a.items = items, a.items_prefilled = 1;
  check(lib.moe_grouped_int4_mlp(&a, st), "anna_mi_moe_grouped_int4_mlp");
  check(lib.moe_combine(w0 + o_y, dt, H, pos, T, top_k, ptr(out), st), "anna_mi_moe_combine");
  return out;
}

}  // namespace

#ifndef ANNA_MI_SOURCE_HASH
#define ANNA_MI_SOURCE_HASH "unstamped"
#endif

PYBIND11_MODULE(_torch_host, m) {
  const auto no_gil = py::call_guard<py::gil_scoped_release>();
  m.def("source_hash", [] { return std::string(ANNA_MI_SOURCE_HASH); });
  m.def("bind", &bind);
  m.def("int4_linear", &int4_linear, no_gil, py::arg("x"), py::arg("qweight"), py::arg("qscale"), py::arg("qzeros"),
        py::arg("bias"), py::arg("group"), py::arg("out_features"), py::arg("compute"), py::arg("stream"),
        py::arg("strategies") = true);
  m.def("decode_rows", &decode_rows, no_gil);
  m.def("decode_pool", &decode_pool, no_gil);
  m.def("tq_store", &tq_store, no_gil);
  m.def("moe_block", &moe_block, no_gil);
}
