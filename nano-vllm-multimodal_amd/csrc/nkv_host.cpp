// Per-call host path of the hip backend's store, gather and attention.
//
// The reference's SDPA decode calls its backend's gather twice per request
// per layer (nanovllm/layers/attention.py:284-300) and its store once per
// layer (attention.py:87-93).  Each call validates its inputs
// (nanovllm/layers/paged_kv/base.py:75-151) and launches one kernel.  On
// MI355X the launch alone costs about 3 us of host time, so Python around
// it (argument checks, the output allocation, a ctypes call) was most of a
// call.  This module runs the same checks, in the same order and with the
// same ValueError messages as nanokv.paged_kv.base.check_store_inputs /
// check_gather_inputs, allocates the gather's output with torch's caching
// allocator, and calls the library's C ABI (include/nanokv.h) directly.
//
// torch is plumbing here: it unpacks the tensors and allocates; every byte
// is moved by the HIP library.  The module does not link libnanokv.so: the
// Python loader hands it the entry points of the library it loaded, so a
// library chosen at run time is the one that runs.  The stream is the
// caller's current stream, passed in as a hipStream_t integer.
#include <torch/extension.h>

#include <algorithm>
#include <cctype>
#include <cstdint>
#include <cstdlib>
#include <string>

#include "nanokv.h"

#ifndef NKV_HOST_BUILD_ID
#define NKV_HOST_BUILD_ID "unfingerprinted"
#endif

namespace {

namespace py = pybind11;

using StoreFn = int (*)(const void*, const void*, void*, void*, const int32_t*, int64_t, int64_t,
                        int64_t, int64_t, int64_t, int32_t, void*);
using GatherFn = int (*)(const void*, const int32_t*, int64_t, int64_t, int64_t, int64_t, int64_t,
                         int32_t, void*, void*);
using LastErrorFn = const char* (*)();

StoreFn g_store = nullptr;
GatherFn g_gather = nullptr;
LastErrorFn g_last_error = nullptr;

[[noreturn]] void value_error(const std::string& what) { throw py::value_error(what); }

void require_bound() {
  if (g_store == nullptr || g_gather == nullptr || g_last_error == nullptr) {
    throw std::runtime_error("nanokv host path: bind() the library's entry points first");
  }
}

// base.py:68-72: index values in host memory are always range-checked;
// device-resident ones only when NANOVLLM_PAGED_KV_VALIDATE_INDICES is one
// of 1 / true / yes / on (read on every call, as the reference does).
bool index_values_checked(const at::Tensor& t) {
  if (!t.is_cuda()) return true;
  const char* raw = std::getenv("NANOVLLM_PAGED_KV_VALIDATE_INDICES");
  std::string flag = raw != nullptr ? raw : "0";
  const char* space = " \t\n\r\f\v";
  const size_t first = flag.find_first_not_of(space);
  flag = first == std::string::npos ? "" : flag.substr(first, flag.find_last_not_of(space) - first + 1);
  for (char& c : flag) c = static_cast<char>(std::tolower(static_cast<unsigned char>(c)));
  return flag == "1" || flag == "true" || flag == "yes" || flag == "on";
}

int32_t dtype_code(at::ScalarType type) {
  switch (type) {
    case at::kHalf:
      return NKV_DTYPE_FLOAT16;
    case at::kBFloat16:
      return NKV_DTYPE_BFLOAT16;
    case at::kFloat:
      return NKV_DTYPE_FLOAT32;
    default:
      throw std::runtime_error(std::string("nanokv paged KV ops support float16, bfloat16 and "
                                           "float32, not ") + c10::toString(type));
  }
}

void check_status(int status, const char* what) {
  if (status != 0) {
    throw std::runtime_error(std::string(what) + " failed (nkv status " + std::to_string(status) +
                             "): " + g_last_error());
  }
}

// The checks of base.py:75-114 (nanokv.paged_kv.base.check_store_inputs).
void check_store(const at::Tensor& key, const at::Tensor& value, const at::Tensor& key_cache,
                 const at::Tensor& value_cache, const at::Tensor& slot_mapping) {
  if (key.dim() != 3 || value.dim() != 3 || key.sizes() != value.sizes()) {
    value_error("key and value must have matching shape [tokens, kv_heads, head_dim]");
  }
  if (key.stride(-1) != 1 || value.stride(-1) != 1) {
    value_error("key and value inner dimensions must be contiguous");
  }
  if (key_cache.dim() != 4 || value_cache.dim() != 4 || key_cache.sizes() != value_cache.sizes()) {
    value_error("key and value cache shape must match [blocks, block, kv_heads, head_dim]");
  }
  if (key_cache.size(2) != key.size(1) || key_cache.size(3) != key.size(2)) {
    value_error("cache shape does not match key/value kv_heads and head_dim");
  }
  const at::Device device = key.device();
  if (value.device() != device || key_cache.device() != device || value_cache.device() != device ||
      slot_mapping.device() != device) {
    value_error("all paged KV Store tensors must be on the same device");
  }
  const at::ScalarType type = key.scalar_type();
  if (value.scalar_type() != type || key_cache.scalar_type() != type ||
      value_cache.scalar_type() != type) {
    value_error("key, value, and caches must have matching dtype");
  }
  if (slot_mapping.scalar_type() != at::kInt || slot_mapping.dim() != 1) {
    value_error("slot_mapping must be a one-dimensional int32 tensor");
  }
  if (slot_mapping.size(0) != key.size(0)) {
    value_error("slot_mapping length must equal the number of input tokens");
  }
  if (!slot_mapping.is_contiguous()) value_error("slot_mapping must be contiguous");
  if (key.size(0) > 0 && index_values_checked(slot_mapping)) {
    const int64_t num_slots = key_cache.size(0) * key_cache.size(1);
    if (((slot_mapping < -1) | (slot_mapping >= num_slots)).any().item<bool>()) {
      value_error("slot_mapping contains a slot outside [-1, " + std::to_string(num_slots) + ")");
    }
  }
}

// The checks of base.py:117-151 (nanokv.paged_kv.base.check_gather_inputs).
void check_gather(const at::Tensor& cache, const at::Tensor& table, int64_t sequence_length) {
  if (cache.dim() != 4) value_error("cache must have shape [blocks, block, kv_heads, head_dim]");
  if (cache.stride(-1) != 1) value_error("cache inner dimensions must be contiguous");
  if (table.scalar_type() != at::kInt || table.dim() != 1) {
    value_error("block_table must be a one-dimensional int32 tensor");
  }
  if (table.device() != cache.device()) {
    value_error("cache and block_table must be on the same device");
  }
  if (!table.is_contiguous()) value_error("block_table must be contiguous");
  if (sequence_length < 0) value_error("sequence_length must be non-negative");
  const int64_t block_size = cache.size(1);
  const int64_t required = (sequence_length + block_size - 1) / block_size;
  if (table.size(0) < required) {
    value_error("block_table does not cover the requested sequence length");
  }
  if (required > 0 && index_values_checked(table)) {
    const at::Tensor used = table.slice(0, 0, required);
    if (((used < 0) | (used >= cache.size(0))).any().item<bool>()) {
      value_error("block_table contains an invalid physical block");
    }
  }
}

void store(const at::Tensor& key_in, const at::Tensor& value_in, const at::Tensor& key_cache,
           const at::Tensor& value_cache, const at::Tensor& slot_mapping, int64_t stream) {
  check_store(key_in, value_in, key_cache, value_cache, slot_mapping);
  if (!key_in.is_cuda()) value_error("HIP Paged KV Store requires ROCm device tensors");
  require_bound();
  if (!key_cache.is_contiguous() || !value_cache.is_contiguous()) {
    value_error("paged KV HIP Store requires contiguous [blocks, block, kv_heads, head_dim] caches");
  }
  const int64_t tokens = key_in.size(0);
  if (tokens == 0) return;
  const int32_t code = dtype_code(key_in.scalar_type());
  // The kernel addresses a token's [kv_heads, head_dim] as one contiguous
  // row through the token stride; a head-strided view is compacted first.
  const bool strided = key_in.size(1) > 1;
  const at::Tensor key =
      strided && key_in.stride(1) != key_in.size(2) ? key_in.contiguous() : key_in;
  const at::Tensor value =
      strided && value_in.stride(1) != value_in.size(2) ? value_in.contiguous() : value_in;
  check_status(g_store(key.data_ptr(), value.data_ptr(), key_cache.data_ptr(),
                       value_cache.data_ptr(), slot_mapping.data_ptr<int32_t>(), tokens,
                       key.stride(0), value.stride(0), key.size(1) * key.size(2),
                       key_cache.size(0) * key_cache.size(1), code,
                       reinterpret_cast<void*>(stream)),
               "nanovllm_paged_kv::store");
}

at::Tensor gather(const at::Tensor& cache, const at::Tensor& table, int64_t sequence_length,
                  int64_t stream) {
  check_gather(cache, table, sequence_length);
  if (!cache.is_cuda()) value_error("HIP Paged KV Gather requires ROCm device tensors");
  require_bound();
  if (!cache.is_contiguous()) {
    value_error("paged KV HIP Gather requires contiguous [blocks, block, kv_heads, head_dim] caches");
  }
  at::Tensor out = at::empty({sequence_length, cache.size(2), cache.size(3)}, cache.options());
  if (sequence_length == 0) return out;
  const int32_t code = dtype_code(cache.scalar_type());
  check_status(g_gather(cache.data_ptr(), table.data_ptr<int32_t>(), table.size(0),
                        sequence_length, cache.size(1), cache.size(2) * cache.size(3),
                        cache.size(0), code, out.data_ptr(), reinterpret_cast<void*>(stream)),
               "nanovllm_paged_kv::gather");
  return out;
}

// ------------------------------------------------------------- attention
//
// One layer's attention call, whole, for the calls an engine makes: every
// tensor as the kernels take it.  A call that any check of the Python path
// would refuse, convert or look into returns None instead, and the Python
// path serves it (or raises), so nothing is decided twice.  Per call the
// Python checks, allocations and ctypes conversions were 17-20 us of host
// time, more than the kernels of a short context take.
using PlanCapacityFn = int64_t (*)(int64_t, int64_t, int64_t);
using WorkspaceFn = int64_t (*)(int64_t, int64_t, int64_t);
using DecodeFn = decltype(&nkv_paged_attention_decode_total);
using PrefillPlanFn = decltype(&nkv_build_prefill_plan);
using PrefillFn = decltype(&nkv_paged_attention_prefill_split);
using VarlenFn = decltype(&nkv_varlen_attention_prefill);

PlanCapacityFn g_decode_capacity = nullptr;
WorkspaceFn g_decode_workspace = nullptr;
DecodeFn g_decode = nullptr;
PlanCapacityFn g_prefill_capacity = nullptr;
PrefillPlanFn g_prefill_plan = nullptr;
WorkspaceFn g_prefill_workspace = nullptr;
PrefillFn g_prefill = nullptr;
VarlenFn g_varlen = nullptr;

constexpr int64_t kDim = 128;

bool on(const at::Tensor& t, const at::Device& device) { return t.device() == device; }
bool int32_vector(const at::Tensor& t, const at::Device& device) {
  return t.scalar_type() == at::kInt && t.dim() == 1 && t.is_contiguous() && on(t, device);
}
bool int32_matrix(const at::Tensor& t, const at::Device& device) {
  return t.scalar_type() == at::kInt && t.dim() == 2 && t.is_contiguous() && on(t, device);
}
bool half_type(at::ScalarType type) { return type == at::kHalf || type == at::kBFloat16; }
// [rows, heads, 128] with each row's heads in one run.
bool head_rows(const at::Tensor& t, at::ScalarType type, const at::Device& device) {
  return t.dim() == 3 && t.scalar_type() == type && on(t, device) && t.size(2) == kDim &&
         t.stride(2) == 1 && t.stride(1) == kDim;
}
bool caches(const at::Tensor& k, const at::Tensor& v, at::ScalarType type, const at::Device& device) {
  return k.dim() == 4 && k.sizes() == v.sizes() && k.scalar_type() == type && v.scalar_type() == type &&
         on(k, device) && on(v, device) && k.is_contiguous() && v.is_contiguous() && k.size(2) > 0 &&
         k.size(3) == kDim;
}
// The output to write: the caller's, or a new one; undefined when the
// caller's is not one the kernels write as it is.
at::Tensor output_for(const at::Tensor& q, const c10::optional<at::Tensor>& out) {
  if (!out.has_value()) return at::empty_like(q);
  if (out->sizes() != q.sizes() || !head_rows(*out, q.scalar_type(), q.device())) return {};
  return *out;
}
at::Tensor bytes_on(int64_t bytes, const at::Tensor& like) {
  return at::empty({bytes}, like.options().dtype(at::kByte));
}
// Room for the partials of a prefill launch that cuts its keys.  Undefined
// where there is none to need, or to have: the launch then cuts nothing.
at::Tensor partials_on(int64_t bytes, const at::Tensor& like) {
  if (bytes <= 0) return {};
  try {
    return bytes_on(bytes, like);
  } catch (const c10::OutOfMemoryError&) {
    return {};
  }
}
void* data_or_null(const at::Tensor& t) { return t.size(0) > 0 ? t.data_ptr() : nullptr; }

// The offsets are only checked (the plan holds what the kernels need);
// callers that built the plan from the lengths have none.
// The checked part of a call, which allocates and launches and may wait for
// either, without the interpreter lock, as in torch's own calls and through
// ctypes; None where it gives no tensor.
template <typename Launch>
py::object run_unlocked(Launch&& launch) {
  at::Tensor out;
  {
    py::gil_scoped_release unlocked;
    out = launch();
  }
  if (!out.defined()) return py::none();
  return py::cast(out);
}

py::object decode(const at::Tensor& q, const at::Tensor& key_cache, const at::Tensor& value_cache,
                  const at::Tensor& tables, const c10::optional<at::Tensor>& cu_seqlens_k,
                  const at::Tensor& plan, const at::Tensor& first_part, int64_t total_tokens,
                  double scale, const c10::optional<at::Tensor>& out_in, int64_t stream) {
  const at::Device device = q.device();
  const at::ScalarType type = q.scalar_type();
  if (g_decode == nullptr || !q.is_cuda() || !half_type(type) || !head_rows(q, type, device) ||
      !caches(key_cache, value_cache, type, device) || !int32_matrix(tables, device) ||
      !int32_matrix(plan, device) || !int32_vector(first_part, device) || total_tokens < 0 ||
      index_values_checked(tables)) {
    return py::none();
  }
  const int64_t seqs = q.size(0);
  if (cu_seqlens_k.has_value() &&
      (!int32_vector(*cu_seqlens_k, device) || cu_seqlens_k->size(0) != seqs + 1)) {
    return py::none();
  }
  if (seqs == 0 || tables.size(0) != seqs || first_part.size(0) != seqs + 1 || plan.size(1) != 4 ||
      plan.size(0) < g_decode_capacity(total_tokens, seqs, key_cache.size(1))) {
    return py::none();
  }
  return run_unlocked([&]() -> at::Tensor {
    const at::Tensor out = output_for(q, out_in);
    if (!out.defined()) return {};
    const int64_t capacity = plan.size(0);
    const int64_t need = std::max<int64_t>(g_decode_workspace(capacity, q.size(1), kDim), 16);
    const at::Tensor workspace = bytes_on(need, q);
    check_status(g_decode(q.data_ptr(), q.stride(0), key_cache.data_ptr(), value_cache.data_ptr(),
                          tables.data_ptr<int32_t>(), tables.size(1), data_or_null(plan), capacity,
                          first_part.data_ptr<int32_t>(), seqs, key_cache.size(2), q.size(1), kDim,
                          key_cache.size(1), key_cache.size(0), static_cast<float>(scale),
                          dtype_code(type), workspace.data_ptr(), need, out.data_ptr(), out.stride(0),
                          total_tokens, reinterpret_cast<void*>(stream)),
                 "nanovllm_paged_kv::paged_attention_decode");
    return out;
  });
}

// A prefill plan for these offsets, or undefined where the head layout has none.
at::Tensor prefill_plan(const at::Tensor& q, int64_t kv_heads, const at::Tensor& cu_q,
                        const at::Tensor& cu_k, int64_t stream) {
  const int64_t seqs = cu_q.size(0) - 1, group = q.size(1) / kv_heads;
  const int64_t capacity = g_prefill_capacity(q.size(0), seqs, group);
  if (capacity == 0) return {};
  const at::Tensor plan = at::empty({capacity, 4}, cu_q.options());
  check_status(g_prefill_plan(cu_q.data_ptr<int32_t>(), cu_k.data_ptr<int32_t>(), seqs, group,
                              plan.data_ptr(), capacity, reinterpret_cast<void*>(stream)),
               "nanovllm_paged_kv::build_prefill_plan");
  return plan;
}

py::object prefill(const at::Tensor& q, const at::Tensor& key_cache, const at::Tensor& value_cache,
                   const at::Tensor& tables, const at::Tensor& cu_q, const at::Tensor& cu_k,
                   const c10::optional<at::Tensor>& plan_in, double scale,
                   const c10::optional<at::Tensor>& out_in, int64_t stream) {
  const at::Device device = q.device();
  const at::ScalarType type = q.scalar_type();
  if (g_prefill == nullptr || !q.is_cuda() || !half_type(type) || !head_rows(q, type, device) ||
      !caches(key_cache, value_cache, type, device) || !int32_matrix(tables, device) ||
      !int32_vector(cu_q, device) || !int32_vector(cu_k, device) || cu_q.size(0) != cu_k.size(0) ||
      cu_q.size(0) < 2 || tables.size(0) != cu_q.size(0) - 1 || index_values_checked(cu_k)) {
    return py::none();
  }
  const int64_t seqs = cu_q.size(0) - 1, kv_heads = key_cache.size(2);
  if (plan_in.has_value() &&
      (!int32_matrix(*plan_in, device) || plan_in->size(1) != 4 || q.size(1) % kv_heads != 0 ||
       plan_in->size(0) < g_prefill_capacity(q.size(0), seqs, q.size(1) / kv_heads))) {
    return py::none();
  }
  return run_unlocked([&]() -> at::Tensor {
    const at::Tensor out = output_for(q, out_in);
    if (!out.defined()) return {};
    const at::Tensor plan = plan_in.has_value() ? *plan_in : prefill_plan(q, kv_heads, cu_q, cu_k, stream);
    if (!plan.defined()) return {};
    const int64_t need = g_prefill_workspace(plan.size(0), kv_heads, tables.size(1) * key_cache.size(1));
    const at::Tensor workspace = partials_on(need, q);
    check_status(g_prefill(q.data_ptr(), q.stride(0), key_cache.data_ptr(), value_cache.data_ptr(),
                           tables.data_ptr<int32_t>(), tables.size(1), cu_q.data_ptr<int32_t>(),
                           cu_k.data_ptr<int32_t>(), data_or_null(plan), plan.size(0), seqs, kv_heads,
                           q.size(1), kDim, key_cache.size(1), key_cache.size(0),
                           static_cast<float>(scale), dtype_code(type), out.data_ptr(), out.stride(0),
                           workspace.defined() ? workspace.data_ptr() : nullptr, need,
                           reinterpret_cast<void*>(stream)),
                 "nanovllm_paged_kv::paged_attention_prefill");
    return out;
  });
}

// Keys and values back to back, read where they lie: rows of [kv_heads, 128]
// each in one run, 16-byte aligned.
py::object varlen(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v,
                  const at::Tensor& cu_q, const at::Tensor& cu_k, int64_t max_seqlen_k, double scale,
                  int64_t stream) {
  const at::Device device = q.device();
  const at::ScalarType type = q.scalar_type();
  if (g_varlen == nullptr || !q.is_cuda() || !half_type(type) || !head_rows(q, type, device) ||
      !head_rows(k, type, device) || !head_rows(v, type, device) || k.sizes() != v.sizes() ||
      k.size(0) == 0 || k.size(1) == 0 || !int32_vector(cu_q, device) || !int32_vector(cu_k, device) ||
      cu_q.size(0) != cu_k.size(0) || cu_q.size(0) < 2 || index_values_checked(cu_k)) {
    return py::none();
  }
  for (const at::Tensor* t : {&k, &v}) {
    if (t->stride(0) < kDim * t->size(1) || t->stride(0) % 8 != 0 ||
        reinterpret_cast<uintptr_t>(t->data_ptr()) % 16 != 0) {
      return py::none();
    }
  }
  return run_unlocked([&]() -> at::Tensor {
    const int64_t seqs = cu_q.size(0) - 1, kv_heads = k.size(1);
    const at::Tensor plan = prefill_plan(q, kv_heads, cu_q, cu_k, stream);
    if (!plan.defined()) return {};
    const at::Tensor out = at::empty_like(q);
    const int64_t longest = std::max<int64_t>(max_seqlen_k, 1);
    const int64_t need = g_prefill_workspace(plan.size(0), kv_heads, longest);
    const at::Tensor workspace = partials_on(need, q);
    check_status(g_varlen(q.data_ptr(), q.stride(0), k.data_ptr(), k.stride(0), v.data_ptr(),
                          v.stride(0), k.size(0), longest, cu_q.data_ptr<int32_t>(),
                          cu_k.data_ptr<int32_t>(), plan.data_ptr(), plan.size(0), seqs, kv_heads,
                          q.size(1), kDim, static_cast<float>(scale), dtype_code(type), out.data_ptr(),
                          out.stride(0), workspace.defined() ? workspace.data_ptr() : nullptr, need,
                          reinterpret_cast<void*>(stream)),
                 "nanovllm_paged_kv::varlen_attention_prefill");
    return out;
  });
}

void bind_attention(uintptr_t decode_capacity, uintptr_t decode_workspace, uintptr_t decode_fn,
                    uintptr_t prefill_capacity, uintptr_t prefill_plan_fn, uintptr_t prefill_workspace,
                    uintptr_t prefill_fn, uintptr_t varlen_fn) {
  g_decode_capacity = reinterpret_cast<PlanCapacityFn>(decode_capacity);
  g_decode_workspace = reinterpret_cast<WorkspaceFn>(decode_workspace);
  g_decode = reinterpret_cast<DecodeFn>(decode_fn);
  g_prefill_capacity = reinterpret_cast<PlanCapacityFn>(prefill_capacity);
  g_prefill_plan = reinterpret_cast<PrefillPlanFn>(prefill_plan_fn);
  g_prefill_workspace = reinterpret_cast<WorkspaceFn>(prefill_workspace);
  g_prefill = reinterpret_cast<PrefillFn>(prefill_fn);
  g_varlen = reinterpret_cast<VarlenFn>(varlen_fn);
}

void bind(uintptr_t store_fn, uintptr_t gather_fn, uintptr_t last_error_fn) {
  g_store = reinterpret_cast<StoreFn>(store_fn);
  g_gather = reinterpret_cast<GatherFn>(gather_fn);
  g_last_error = reinterpret_cast<LastErrorFn>(last_error_fn);
}

}  // namespace

PYBIND11_MODULE(_nkv_host, m) {
  m.doc() = "Per-call host path of the nanokv hip backend's store, gather and attention";
  m.def("bind", &bind, "set the library entry points (nkv_store, nkv_gather, nkv_last_error)");
  m.def("bind_attention", &bind_attention, "set the library's attention entry points");
  m.def("decode", &decode, "planned decode attention; None when the general path has to look at it");
  m.def("prefill", &prefill, "paged prefill attention; None when the general path has to look at it");
  m.def("varlen", &varlen, "prefill attention over keys back to back; None when the general path "
                           "has to look at it");
  m.def("store", &store, "validated store launch on a stream");
  m.def("gather", &gather, "validated gather launch on a stream; returns the new tensor");
  m.def("check_store", &check_store, "the store validator's checks (no launch)");
  m.def("check_gather", &check_gather, "the gather validator's checks (no launch)");
  m.def("build_id", []() { return std::string(NKV_HOST_BUILD_ID); });
}
