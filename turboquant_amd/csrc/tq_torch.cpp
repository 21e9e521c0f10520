// tq_torch.cpp -- torch's side of the C ABI: the calls of turboquant_amd/ops.py
// from C++, and the kernels of the turboquant_write / turboquant_v5 ops behind
// the CUDA (= HIP on ROCm) dispatch key.
//
// A small call is host-bound: in Python, the checks, the tensor addresses, the
// device and stream look-ups and the ctypes call of a write took 13 us around
// a 4 us launch.  Every function here looks at the same conditions as its
// counterpart in ops.py and launches if all of them hold; if anything is out
// of the ordinary (a refused argument, an unaligned tensor that has to be
// copied, a tensor subclass, an error from the library) it does nothing and
// says so, and ops.py goes through its own checks, which raise, copy or launch
// as they always did.  So ops.py stays the one place that defines what is
// accepted and how it is refused.
#include <ATen/ops/empty.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/utils/pybind.h>
#include <torch/library.h>

#include <array>
#include <cmath>
#include <optional>
#include <tuple>
#include <vector>

#include "../../include/turboquant_amd.h"

namespace {

namespace py = pybind11;
using at::Tensor;
using OptTensor = std::optional<Tensor>;

// a plain tensor (no subclass or functional wrapper) on GPU `dev`
bool on(const Tensor& t, c10::Device dev) {
  if (!t.defined() || !t.is_cuda() || t.device() != dev) return false;
  constexpr c10::DispatchKeySet wrapped({c10::DispatchKey::Python, c10::DispatchKey::Functionalize,
                                         c10::DispatchKey::FuncTorchBatched,
                                         c10::DispatchKey::FuncTorchGradWrapper});
  return !t.key_set().has_any(wrapped);
}

template <class T>
const T* cptr(const Tensor& t) {
  return static_cast<const T*>(t.const_data_ptr());
}

bool aligned(const Tensor& t, uintptr_t n) { return (uintptr_t)t.const_data_ptr() % n == 0; }

tq_stream_t stream_of(c10::Device dev) {
  return reinterpret_cast<tq_stream_t>(c10::hip::getCurrentHIPStream(dev.index()).stream());
}

bool is_i32(const Tensor& t, c10::Device dev) {
  return on(t, dev) && t.scalar_type() == at::kInt && t.is_contiguous();
}

bool is_f32(const Tensor& t, c10::Device dev) {
  return on(t, dev) && t.scalar_type() == at::kFloat && t.is_contiguous();
}

int dtype_code(at::ScalarType t) {
  return t == at::kFloat ? TQ_F32 : t == at::kHalf ? TQ_F16 : t == at::kBFloat16 ? TQ_BF16 : -1;
}

bool is_half(int code) { return code == TQ_F16 || code == TQ_BF16; }

// the paged cache [2, num_blocks, block_size, H, ebs]
struct Cache {
  const uint8_t* k = nullptr;
  const uint8_t* v = nullptr;
  int64_t num_blocks = 0, block_size = 16, heads = 0, ebs = 0;
};
bool cache_of(const Tensor& t, c10::Device dev, Cache& c) {
  if (!on(t, dev) || t.dim() != 5 || t.size(0) != 2 || !t.is_contiguous()) return false;
  c.num_blocks = t.size(1);
  c.block_size = t.size(2);
  c.heads = t.size(3);
  c.ebs = t.size(4) * t.element_size();
  c.k = static_cast<const uint8_t*>(t.const_data_ptr());
  c.v = c.k + c.num_blocks * c.block_size * c.heads * c.ebs;
  return true;
}

// signs fp32 [>= padded_dim] contiguous, or none
bool signs_of(const OptTensor& t, int64_t padded_dim, c10::Device dev, const float*& p) {
  p = nullptr;
  if (!t.has_value() || t->numel() == 0) return true;
  if (!is_f32(*t, dev) || t->numel() < padded_dim) return false;
  p = cptr<float>(*t);
  return true;
}

// ops.quantize_write_kv_cache
bool write_cache(const Tensor& kv_cache, const Tensor& key, const Tensor& value,
                 const Tensor& signs, const Tensor& slots, int64_t head_dim, int64_t padded_dim) {
  const c10::Device dev = kv_cache.device();
  Cache c;
  const float* sp = nullptr;
  if (!cache_of(kv_cache, dev, c) || c.ebs % 16 != 0 || !on(key, dev) || !on(value, dev) ||
      !is_i32(slots, dev) || key.dim() != 3 || value.sizes() != key.sizes() ||
      value.scalar_type() != key.scalar_type() ||
      dtype_code(key.scalar_type()) < 0 || key.size(2) < head_dim || key.stride(2) != 1 ||
      value.stride(2) != 1 || key.size(1) != c.heads || !signs_of(signs, padded_dim, dev, sp) || !sp)
    return false;
  const int64_t n = std::min(key.size(0), slots.numel());
  if (n == 0) return true;
  const c10::DeviceGuard guard(dev);
  return tq_quantize_write_kv_cache(
             const_cast<uint8_t*>(c.k), const_cast<uint8_t*>(c.v), key.const_data_ptr(),
             value.const_data_ptr(), dtype_code(key.scalar_type()), key.stride(0), key.stride(1),
             value.stride(0), value.stride(1), sp, cptr<int32_t>(slots), n, c.heads,
             head_dim, padded_dim, c.block_size, c.ebs, c.num_blocks, stream_of(dev)) == 0;
}

// ops.decode_paged_balanced (rows: decode_paged_balanced_rows)
bool decode_balanced(const Tensor& q, const Tensor& kv_cache, const Tensor& indices,
                     const Tensor& indptr, const Tensor& seq_lens, int64_t num_kv_heads,
                     int64_t head_dim, int64_t padded_dim, double sm_scale, const OptTensor& signs,
                     const Tensor& o, const Tensor& partition_o, const Tensor& partition_lse,
                     const Tensor& split_indptr, bool rows) {
  const c10::Device dev = q.device();
  Cache c;
  const float* sp = nullptr;
  const int64_t row_dim = rows ? head_dim : padded_dim;
  if (!on(q, dev) || q.dim() != 3 || q.size(2) != row_dim || q.stride(2) != 1 ||
      !is_i32(indices, dev) || !is_i32(indptr, dev) || !is_i32(seq_lens, dev) ||
      !is_i32(split_indptr, dev) || !on(o, dev) || !o.is_contiguous() || o.sizes() != q.sizes() ||
      !cache_of(kv_cache, dev, c) || c.heads != num_kv_heads ||
      !signs_of(signs, padded_dim, dev, sp))
    return false;
  const int64_t b = q.size(0), hq = q.size(1);
  const int qt = dtype_code(q.scalar_type()), ot = dtype_code(o.scalar_type());
  if (rows ? !is_half(qt) || !is_half(ot) : qt != TQ_F16 || ot != TQ_F16) return false;
  if (seq_lens.numel() < b || indptr.numel() < b || split_indptr.numel() < b + 2 ||
      !is_f32(partition_o, dev) || partition_o.dim() != 3 || partition_o.size(1) != hq ||
      partition_o.size(2) != padded_dim || !is_f32(partition_lse, dev) ||
      partition_lse.numel() < partition_o.size(0) * hq)
    return false;
  const c10::DeviceGuard guard(dev);
  const int32_t* ip = cptr<int32_t>(indices);
  const int32_t* pp = cptr<int32_t>(indptr);
  const int32_t* lp = cptr<int32_t>(seq_lens);
  const int32_t max_rows = (int32_t)partition_o.size(0);
  float* po = partition_o.data_ptr<float>();
  float* pl = partition_lse.data_ptr<float>();
  int32_t* sr = split_indptr.data_ptr<int32_t>();
  const tq_stream_t st = stream_of(dev);
  if (rows && (row_dim != padded_dim || qt != TQ_F16 || ot != TQ_F16))
    return tq_decode_paged_balanced_rows(
               q.const_data_ptr(), q.stride(0), q.stride(1), qt, c.k, c.v, ip, pp, lp, b, hq,
               num_kv_heads, head_dim, padded_dim, c.block_size, c.ebs, c.num_blocks,
               (float)sm_scale, sp, max_rows, po, pl, sr, o.data_ptr(), ot, st) == 0;
  return tq_decode_paged_balanced(q.const_data_ptr(), q.stride(0), q.stride(1), c.k, c.v, ip, pp,
                                  lp, b, hq, num_kv_heads, head_dim, padded_dim, c.block_size,
                                  c.ebs, c.num_blocks, (float)sm_scale, sp, max_rows, po, pl, sr,
                                  o.data_ptr(), st) == 0;
}

// -------------------------------------------------------------------- prefill

using Request = std::array<int32_t, 5>;

std::array<std::vector<int32_t>, 5> columns(const std::vector<Request>& reqs) {
  std::array<std::vector<int32_t>, 5> c;
  for (auto& v : c) v.reserve(reqs.size());
  for (const Request& r : reqs)
    for (int i = 0; i < 5; i++) c[i].push_back(r[i]);
  return c;
}

// ops.prefill_attention_batch
bool prefill_batch(const Tensor& q, const Tensor& o, const std::vector<Request>& reqs,
                   int64_t num_kv_heads, int64_t head_dim, int64_t padded_dim, double sm_scale,
                   const OptTensor& k, const OptTensor& v, const OptTensor& k2,
                   const OptTensor& v2) {
  const c10::Device dev = q.device();
  const int qt = dtype_code(q.scalar_type()), ot = dtype_code(o.scalar_type());
  if (!on(q, dev) || !on(o, dev) || q.dim() != 3 || o.sizes() != q.sizes() ||
      q.size(2) != head_dim || !is_half(qt) || !is_half(ot) || q.stride(2) != 1 ||
      o.stride(2) != 1 || k.has_value() != v.has_value() || k2.has_value() != v2.has_value() ||
      reqs.empty())
    return false;
  for (const OptTensor* t : {&k, &v, &k2, &v2})
    if (t->has_value() &&
        (!on(**t, dev) || (*t)->scalar_type() != at::kHalf || (*t)->dim() != 3 ||
         (*t)->stride(2) != 1 || (*t)->size(1) != num_kv_heads || (*t)->size(2) != padded_dim))
      return false;
  if ((k.has_value() && k->size(0) != v->size(0)) ||
      (k2.has_value() && (k2->size(0) != v2->size(0) || k2->strides() != v2->strides())))
    return false;
  for (const Request& r : reqs) {  // q_start, q_len, kv_start, kv_len, source
    const OptTensor& kv = r[4] ? k2 : k;
    if (r[0] < 0 || r[1] < 0 || (int64_t)r[0] + r[1] > q.size(0) || !kv.has_value() || r[2] < 0 ||
        r[3] < r[1] || (int64_t)r[2] + r[3] > kv->size(0))
      return false;
  }
  const auto c = columns(reqs);
  const int32_t n = (int32_t)reqs.size(), hq = (int32_t)q.size(1);
  const c10::DeviceGuard guard(dev);
  const int64_t bytes =
      tq_prefill_batch_workspace_bytes(c[1].data(), c[3].data(), n, hq, (int32_t)padded_dim);
  Tensor ws;
  if (bytes > 0) {
    ws = at::empty({bytes}, q.options().dtype(at::kByte));
    if (!on(ws, dev)) return false;
  }
  const auto ptr = [](const OptTensor& t) -> const void* {
    return t.has_value() ? t->const_data_ptr() : nullptr;
  };
  const auto st = [](const OptTensor& t, int i) { return t.has_value() ? t->stride(i) : 0; };
  return tq_prefill_attention_batch(
             q.const_data_ptr(), q.stride(0), q.stride(1), qt, ptr(k), st(k, 0), st(k, 1), ptr(v),
             st(v, 0), st(v, 1), ptr(k2), ptr(v2), st(k2, 0), st(k2, 1), o.data_ptr(), o.stride(0),
             o.stride(1), ot, c[0].data(), c[1].data(), c[2].data(), c[3].data(), c[4].data(), n,
             hq, num_kv_heads, head_dim, padded_dim, (float)sm_scale,
             bytes > 0 ? ws.data_ptr() : nullptr, bytes, stream_of(dev)) == 0;
}

// ops.prefill_gather
bool prefill_gather(const OptTensor& kv_cache, const OptTensor& table, const Tensor& key,
                    const Tensor& value, const std::vector<Request>& reqs, int64_t head_dim,
                    int64_t padded_dim, const OptTensor& signs, const Tensor& out_k,
                    const Tensor& out_v) {
  const c10::Device dev = key.device();
  const int kt = dtype_code(key.scalar_type());
  const float* sp = nullptr;
  if (!on(key, dev) || !on(value, dev) || kt < 0 || value.scalar_type() != key.scalar_type() ||
      key.dim() != 3 || value.sizes() != key.sizes() || key.size(2) != head_dim ||
      key.stride(2) != 1 || value.stride(2) != 1 || !signs_of(signs, padded_dim, dev, sp) ||
      reqs.empty())
    return false;
  const int64_t h = key.size(1);
  for (const Tensor* t : {&out_k, &out_v})
    if (!on(*t, dev) || t->scalar_type() != at::kHalf || t->dim() != 3 || t->size(1) != h ||
        t->size(2) != padded_dim || !t->is_contiguous())
      return false;
  // context needs the cache and its table; a step without any leaves both to ops.py
  Cache c;
  if (!kv_cache.has_value() || !table.has_value() || !cache_of(*kv_cache, dev, c) ||
      c.heads != h || !on(*table, dev) || table->scalar_type() != at::kInt || table->dim() != 2 ||
      table->stride(1) != 1)
    return false;
  const int64_t rows = std::min(out_k.size(0), out_v.size(0));
  for (const Request& r : reqs)  // table_row, ctx, fresh_start, fresh_len, out_start
    if (r[1] < 0 || r[2] < 0 || r[3] < 0 || r[4] < 0 || (int64_t)r[4] + r[1] + r[3] > rows ||
        (int64_t)r[2] + r[3] > key.size(0) || r[0] < 0 ||
        (r[1] > 0 && (r[0] >= table->size(0) || r[1] > table->size(1) * c.block_size)))
      return false;
  const auto cols = columns(reqs);
  const c10::DeviceGuard guard(dev);
  return tq_prefill_gather(c.k, c.v, cptr<int32_t>(*table), table->stride(0), h,
                           head_dim, padded_dim, c.block_size, c.ebs, c.num_blocks, sp,
                           key.const_data_ptr(), value.const_data_ptr(), kt, key.stride(0),
                           key.stride(1), value.stride(0), value.stride(1), cols[0].data(),
                           cols[1].data(), cols[2].data(), cols[3].data(), cols[4].data(),
                           (int32_t)reqs.size(), out_k.data_ptr(), out_v.data_ptr(),
                           stream_of(dev)) == 0;
}

// -------------------------------------------------- the algorithm library

int64_t codes_per_byte(int64_t bits) { return bits == 3 ? 2 : bits >= 1 && bits <= 4 ? 8 / bits : 0; }

// x fp32 [..., dim], contiguous and 16-byte aligned
bool vectors(const Tensor& x, c10::Device dev) {
  return is_f32(x, dev) && x.dim() >= 1 && x.numel() > 0 && aligned(x, 16);
}

std::vector<int64_t> lead_and(const Tensor& t, int64_t last) {
  std::vector<int64_t> s(t.sizes().begin(), t.sizes().end());
  s.back() = last;
  return s;
}

// host tables padded to 16 entries: the library reads 2^bits of them at most
std::array<float, 16> table16(const std::vector<double>& v) {
  std::array<float, 16> t{};
  for (size_t i = 0; i < v.size() && i < 16; i++) t[i] = (float)v[i];
  return t;
}

using MseCodes = std::optional<std::tuple<Tensor, Tensor>>;
using ProdCodes = std::optional<std::tuple<Tensor, Tensor, Tensor, Tensor>>;

// ops.mse_quantize
MseCodes mse_quantize(const Tensor& x, int64_t padded_dim, int64_t bits, const Tensor& signs,
                      const std::vector<double>& boundaries) {
  const c10::Device dev = x.device();
  const int64_t per = codes_per_byte(bits);
  if (!vectors(x, dev) || per == 0 || !is_f32(signs, dev) || signs.numel() < padded_dim ||
      !aligned(signs, 16) || (int64_t)boundaries.size() != (1 << bits) - 1)
    return std::nullopt;
  const int64_t dim = x.size(-1);
  const c10::DeviceGuard guard(dev);
  const Tensor packed = at::empty(lead_and(x, padded_dim / per), x.options().dtype(at::kByte));
  const Tensor norms = at::empty(x.sizes().slice(0, x.dim() - 1), x.options());
  if (!on(packed, dev) || !on(norms, dev)) return std::nullopt;
  const auto b = table16(boundaries);
  if (tq_mse_quantize(cptr<float>(x), x.numel() / dim, dim, padded_dim, bits,
                      cptr<float>(signs), b.data(), packed.data_ptr<uint8_t>(),
                      norms.data_ptr<float>(), stream_of(dev)) != 0)
    return std::nullopt;
  return std::make_tuple(packed, norms);
}

// packed codes [..., padded_dim / per] with fp32 norms [...] of the same rows
bool codes(const Tensor& packed, const Tensor& norms, int64_t padded_dim, int64_t bits,
           c10::Device dev) {
  const int64_t per = codes_per_byte(bits);
  return per != 0 && on(packed, dev) && packed.scalar_type() == at::kByte && packed.dim() >= 1 &&
         packed.size(-1) == padded_dim / per && packed.is_contiguous() && packed.numel() > 0 &&
         aligned(packed, 16) && is_f32(norms, dev) &&
         norms.sizes() == packed.sizes().slice(0, packed.dim() - 1);
}

// ops.mse_dequantize
OptTensor mse_dequantize(const Tensor& packed, const Tensor& norms, int64_t dim,
                         int64_t padded_dim, int64_t bits, const Tensor& signs,
                         const std::vector<double>& centroids) {
  const c10::Device dev = packed.device();
  if (!codes(packed, norms, padded_dim, bits, dev) || dim < 1 || !is_f32(signs, dev) ||
      signs.numel() < padded_dim || !aligned(signs, 16) ||
      (int64_t)centroids.size() != (1 << bits))
    return std::nullopt;
  const c10::DeviceGuard guard(dev);
  const Tensor out = at::empty(lead_and(packed, dim), norms.options());
  if (!on(out, dev)) return std::nullopt;
  const auto c = table16(centroids);
  if (tq_mse_dequantize(cptr<uint8_t>(packed), cptr<float>(norms),
                        norms.numel(), dim, padded_dim, bits, cptr<float>(signs),
                        c.data(), out.data_ptr<float>(), stream_of(dev)) != 0)
    return std::nullopt;
  return out;
}

bool halves(const Tensor& t, int64_t padded_dim, c10::Device dev) {
  return on(t, dev) && t.scalar_type() == at::kHalf && t.dim() == 2 && t.size(0) == padded_dim &&
         t.size(1) == padded_dim && t.is_contiguous() && aligned(t, 16);
}

// ops.qjl_halves
std::optional<std::tuple<Tensor, Tensor, Tensor, Tensor>> qjl_halves(const Tensor& s,
                                                                     int64_t padded_dim) {
  const c10::Device dev = s.device();
  if (!is_f32(s, dev) || s.dim() != 2 || s.size(0) != s.size(1) || s.size(0) < 1 ||
      s.size(0) > padded_dim || padded_dim > 1024)
    return std::nullopt;
  const c10::DeviceGuard guard(dev);
  const Tensor out = at::empty({4, padded_dim, padded_dim}, s.options().dtype(at::kHalf));
  if (!on(out, dev) || tq_qjl_halves(cptr<float>(s), s.size(0), padded_dim, out.data_ptr(),
                                     stream_of(dev)) != 0)
    return std::nullopt;
  return std::make_tuple(out.select(0, 0), out.select(0, 1), out.select(0, 2), out.select(0, 3));
}

// ops.qjl_operand
std::optional<std::tuple<Tensor, Tensor, Tensor>> qjl_operand(const Tensor& s, int64_t padded_dim,
                                                              bool transposed) {
  const c10::Device dev = s.device();
  if (!is_f32(s, dev) || s.dim() != 2 || s.size(0) != s.size(1) || s.size(0) < 1 ||
      s.size(0) > padded_dim || padded_dim > 1024)
    return std::nullopt;
  const c10::DeviceGuard guard(dev);
  const Tensor out = at::empty({2, padded_dim, padded_dim}, s.options().dtype(at::kHalf));
  const Tensor scale = at::empty({padded_dim}, s.options());
  if (!on(out, dev) || !on(scale, dev) ||
      tq_qjl_operand(cptr<float>(s), s.size(0), padded_dim, transposed, out.data_ptr(),
                     scale.data_ptr<float>(), stream_of(dev)) != 0)
    return std::nullopt;
  return std::make_tuple(out.select(0, 0), out.select(0, 1), scale);
}

// the QJL matrix fp32 [dim, dim], or (lo given) its halves
bool matrix_or_halves(const Tensor& s, const OptTensor& lo, int64_t dim, int64_t padded_dim,
                      bool large, c10::Device dev) {
  if (lo.has_value()) return halves(s, padded_dim, dev) && halves(*lo, padded_dim, dev);
  return !large && is_f32(s, dev) && s.dim() == 2 && s.size(0) == dim && s.size(1) == dim &&
         aligned(s, 16);
}

// ops.prod_quantize_qjl (large: prod_quantize_qjl_ws; without s_lo: prod_quantize_qjl_matrix)
ProdCodes prod_quantize_qjl(const Tensor& x, int64_t padded_dim, int64_t bits, const Tensor& signs,
                            const std::vector<double>& boundaries,
                            const std::vector<double>& centroids, const Tensor& s_hi,
                            const OptTensor& s_lo, bool large) {
  const c10::Device dev = x.device();
  const int64_t per = codes_per_byte(bits);
  if (!vectors(x, dev) || per == 0 || !is_f32(signs, dev) || signs.numel() < padded_dim ||
      !aligned(signs, 16) || !matrix_or_halves(s_hi, s_lo, x.size(-1), padded_dim, large, dev) ||
      (int64_t)boundaries.size() != (1 << bits) - 1 || (int64_t)centroids.size() != (1 << bits))
    return std::nullopt;
  const int64_t dim = x.size(-1), n = x.numel() / dim;
  const c10::DeviceGuard guard(dev);
  const Tensor packed = at::empty(lead_and(x, padded_dim / per), x.options().dtype(at::kByte));
  const Tensor norms = at::empty(x.sizes().slice(0, x.dim() - 1), x.options());
  const Tensor z = at::empty(x.sizes(), x.options().dtype(at::kChar));
  const Tensor rnorm = at::empty(norms.sizes(), x.options());
  const int64_t bytes = large ? tq_prod_workspace_bytes(n, (int32_t)padded_dim) : 0;
  const Tensor ws = bytes > 0 ? at::empty({bytes}, x.options().dtype(at::kByte)) : Tensor();
  if (!on(packed, dev) || !on(norms, dev) || !on(z, dev) || !on(rnorm, dev) ||
      (bytes > 0 && !on(ws, dev)))
    return std::nullopt;
  const auto b = table16(boundaries), c = table16(centroids);
  const int rc =
      large ? tq_prod_quantize_qjl_ws(
                  cptr<float>(x), n, dim, padded_dim, bits,
                  cptr<float>(signs), b.data(), c.data(), s_hi.const_data_ptr(),
                  s_lo->const_data_ptr(), packed.data_ptr<uint8_t>(), norms.data_ptr<float>(),
                  z.data_ptr<int8_t>(), rnorm.data_ptr<float>(),
                  bytes > 0 ? ws.data_ptr() : nullptr, bytes, stream_of(dev))
      : s_lo.has_value()
          ? tq_prod_quantize_qjl(cptr<float>(x), n, dim, padded_dim, bits, cptr<float>(signs),
                                 b.data(), c.data(), s_hi.const_data_ptr(), s_lo->const_data_ptr(),
                                 packed.data_ptr<uint8_t>(), norms.data_ptr<float>(),
                                 z.data_ptr<int8_t>(), rnorm.data_ptr<float>(), stream_of(dev))
          : tq_prod_quantize_qjl_matrix(
                cptr<float>(x), n, dim, padded_dim, bits, cptr<float>(signs), b.data(), c.data(),
                cptr<float>(s_hi), packed.data_ptr<uint8_t>(), norms.data_ptr<float>(),
                z.data_ptr<int8_t>(), rnorm.data_ptr<float>(), stream_of(dev));
  if (rc != 0) return std::nullopt;
  return std::make_tuple(packed, norms, z, rnorm);
}

// ops.prod_dequantize_qjl (large: prod_dequantize_qjl_ws; without st_lo:
// prod_dequantize_qjl_matrix, st_hi S itself)
OptTensor prod_dequantize_qjl(const Tensor& packed, const Tensor& norms, const Tensor& z,
                              const Tensor& rnorm, int64_t dim, int64_t padded_dim, int64_t bits,
                              const Tensor& signs, const std::vector<double>& centroids,
                              const Tensor& st_hi, const OptTensor& st_lo, bool large,
                              const OptTensor& st_scale) {
  const c10::Device dev = packed.device();
  if (!codes(packed, norms, padded_dim, bits, dev) || dim < 1 || !is_f32(rnorm, dev) ||
      rnorm.sizes() != norms.sizes() || !on(z, dev) || z.scalar_type() != at::kChar ||
      z.dim() != packed.dim() || z.size(-1) != dim ||
      z.sizes().slice(0, z.dim() - 1) != norms.sizes() || !z.is_contiguous() || !aligned(z, 16) ||
      !is_f32(signs, dev) || signs.numel() < padded_dim || !aligned(signs, 16) ||
      !matrix_or_halves(st_hi, st_lo, dim, padded_dim, large, dev) ||
      (int64_t)centroids.size() != (1 << bits) ||
      (st_scale.has_value() &&
       (!large || !is_f32(*st_scale, dev) || st_scale->numel() < padded_dim)))
    return std::nullopt;
  const c10::DeviceGuard guard(dev);
  const Tensor out = at::empty(lead_and(packed, dim), norms.options());
  if (!on(out, dev)) return std::nullopt;
  const auto c = table16(centroids);
  const int rc =
      large ? tq_prod_dequantize_qjl_ws(
                  cptr<uint8_t>(packed), cptr<float>(norms), cptr<int8_t>(z), cptr<float>(rnorm),
                  norms.numel(), dim, padded_dim, bits, cptr<float>(signs), c.data(),
                  st_hi.const_data_ptr(), st_lo->const_data_ptr(),
                  st_scale.has_value() ? cptr<float>(*st_scale) : nullptr, out.data_ptr<float>(),
                  stream_of(dev))
      : st_lo.has_value()
          ? tq_prod_dequantize_qjl(
                cptr<uint8_t>(packed), cptr<float>(norms), cptr<int8_t>(z), cptr<float>(rnorm),
                norms.numel(), dim, padded_dim, bits, cptr<float>(signs), c.data(),
                st_hi.const_data_ptr(), st_lo->const_data_ptr(), out.data_ptr<float>(),
                stream_of(dev))
          : tq_prod_dequantize_qjl_matrix(
                cptr<uint8_t>(packed), cptr<float>(norms), cptr<int8_t>(z), cptr<float>(rnorm),
                norms.numel(), dim, padded_dim, bits, cptr<float>(signs), c.data(),
                cptr<float>(st_hi), out.data_ptr<float>(), stream_of(dev));
  if (rc != 0) return std::nullopt;
  return out;
}

// ----------------------------------------------------------- dispatcher kernels

// ops.<name>(args...), with its checks and errors
template <class... A>
void in_python(const char* name, const A&... args) {
  const py::gil_scoped_acquire gil;
  py::module_::import("turboquant_amd.ops").attr(name)(args...);
}

void write_op(const Tensor& kv_cache, const Tensor& key, const Tensor& value, const Tensor& signs,
              const Tensor& slot_mapping, int64_t head_dim, int64_t padded_dim) {
  if (!write_cache(kv_cache, key, value, signs, slot_mapping, head_dim, padded_dim))
    in_python("quantize_write_kv_cache", kv_cache, key, value, signs, slot_mapping, head_dim,
              padded_dim);
}

template <bool ROWS>
void balanced_op(const Tensor& q, const Tensor& kv_cache, const Tensor& indices,
                 const Tensor& indptr, const Tensor& seq_lens, int64_t num_kv_heads,
                 int64_t head_dim, int64_t padded_dim, double sm_scale,
                 const Tensor& hadamard_signs, const Tensor& o_ws, const Tensor& partition_o_ws,
                 const Tensor& partition_lse_ws, const Tensor& split_indptr) {
  if (!decode_balanced(q, kv_cache, indices, indptr, seq_lens, num_kv_heads, head_dim, padded_dim,
                       sm_scale, hadamard_signs, o_ws, partition_o_ws, partition_lse_ws,
                       split_indptr, ROWS))
    in_python(ROWS ? "decode_paged_balanced_rows" : "decode_paged_balanced", q, kv_cache, indices,
              indptr, seq_lens, num_kv_heads, head_dim, padded_dim, sm_scale, hadamard_signs, o_ws,
              partition_o_ws, partition_lse_ws, split_indptr);
}

}  // namespace

TORCH_LIBRARY_IMPL(turboquant_write, CUDA, m) { m.impl("quantize_write_kv_cache", write_op); }

TORCH_LIBRARY_IMPL(turboquant_v5, CUDA, m) {
  m.impl("decode_paged_balanced_ws", balanced_op<false>);
  m.impl("decode_paged_balanced_rows_ws", balanced_op<true>);
}

PYBIND11_MODULE(_tq_torch, m) {
  m.attr("abi_version") = TQ_ABI_VERSION;
  const auto unlocked = py::call_guard<py::gil_scoped_release>();
  m.def("write_cache", &write_cache, unlocked);
  m.def("decode_balanced", &decode_balanced, unlocked);
  m.def("prefill_batch", &prefill_batch, unlocked);
  m.def("prefill_gather", &prefill_gather, unlocked);
  m.def("mse_quantize", &mse_quantize, unlocked);
  m.def("mse_dequantize", &mse_dequantize, unlocked);
  m.def("qjl_halves", &qjl_halves, unlocked);
  m.def("qjl_operand", &qjl_operand, unlocked);
  m.def("prod_quantize_qjl", &prod_quantize_qjl, unlocked);
  m.def("prod_dequantize_qjl", &prod_dequantize_qjl, unlocked);
}
