// The operators' torch kernels (libpiper_torch.so): piper_kernels::piper_attention and
// piper_kernels::sage_attention_2pp on GPU tensors, over the C ABI of libpiper_mi355x.so.
//
// Short calls are bound by the host: at B1 H4 Sq35 Sk67 D64, whose kernels take 13 us, the same two library
// calls from Python, with their argument structs, ten allocations and stream and device queries, take 41 us
// (calls in a row).  Here a call makes two allocations (the output, and one workspace that holds every prepared
// buffer): the whole public call takes 17 us.  The op's definition, its fake and its autograd stay in Python
// (torch.library.custom_op), which also runs calls under an explicit launch plan.
#include <ATen/ATen.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <c10/core/DeviceGuard.h>
#include <torch/library.h>

#include <array>
#include <atomic>
#include <exception>
#include <map>
#include <memory>
#include <mutex>
#include <string>

#include "piper_mi355x.h"

namespace {

enum Operator : int32_t { kPiper = 0, kSage = 1 };

// Launch plans: chosen by the Python package (its frozen tables and heuristics), asked once per shape.
// Returns a plan id, or a negative number after an error.
using PlanSource = int32_t (*)(int32_t op, int64_t batch, int64_t heads, int64_t query_length, int64_t key_length,
                               int64_t head_dim, int32_t is_causal);
std::atomic<PlanSource> g_plan_source{nullptr};
thread_local std::string g_plan_error;  // why the source of this thread's call found no plan

using PlanKey = std::array<int64_t, 7>;
std::mutex g_plans_mutex;
std::map<PlanKey, int32_t> g_plans;
constexpr size_t kMaxPlans = 4096;  // shapes remembered; past it the map starts over

int32_t plan_for(Operator op, const piper_shape& s, bool causal) {
  const PlanKey key{op, s.batch, s.heads, s.query_length, s.key_length, s.head_dim, causal};
  {
    std::lock_guard<std::mutex> lock(g_plans_mutex);
    const auto found = g_plans.find(key);
    if (found != g_plans.end()) return found->second;
  }
  const PlanSource source = g_plan_source.load();
  TORCH_CHECK(source != nullptr, "piper_kernels: no launch-plan source is set");
  g_plan_error.clear();
  // without the lock: the source takes Python's
  const int32_t plan = source(op, s.batch, s.heads, s.query_length, s.key_length, s.head_dim, causal);
  TORCH_CHECK(plan >= 0, "piper_kernels: no launch plan for this shape: ", g_plan_error);
  std::lock_guard<std::mutex> lock(g_plans_mutex);
  if (g_plans.size() >= kMaxPlans) g_plans.clear();
  g_plans.emplace(key, plan);
  return plan;
}

void check(int status, const char* what) {
  TORCH_CHECK(status == PIPER_OK, what, " failed (status ", status, "): ", piper_last_error());
}

int32_t dtype_code(const at::Tensor& t) {
  TORCH_CHECK(t.scalar_type() == at::kHalf || t.scalar_type() == at::kBFloat16,
              "piper_kernels: tensors must use float16 or bfloat16, got ", t.scalar_type());
  return t.scalar_type() == at::kBFloat16 ? PIPER_BFLOAT16 : PIPER_FLOAT16;
}

// Any [B, H, S, D] view whose rows are 16-byte aligned is read in place (the strides of axes of size 1 do
// not count); anything else is copied.  A copy, not contiguous(): that keeps a contiguous view as it is, also
// one that starts between two 16-byte boundaries.
at::Tensor native_input(const at::Tensor& t) {
  bool in_place = (reinterpret_cast<uintptr_t>(t.const_data_ptr()) & 15u) == 0 && t.stride(3) == 1;
  for (int64_t axis = 0; axis < 3; ++axis) in_place = in_place && (t.size(axis) == 1 || t.stride(axis) % 8 == 0);
  return in_place ? t : t.clone(at::MemoryFormat::Contiguous);
}

piper_tensor tensor_arg(const at::Tensor& t) {
  const auto stride = [&](int64_t axis) { return t.size(axis) == 1 ? 0 : t.stride(axis); };
  return piper_tensor{t.const_data_ptr(), stride(0), stride(1), stride(2)};
}

// One allocation handed out in 256-byte steps.
struct Arena {
  int64_t size = 0;
  int64_t take(int64_t bytes) {
    const int64_t offset = size;
    size += (bytes + 255) / 256 * 256;
    return offset;
  }
};

// The kernels read key and value by the query's shape and device, the value by the key's type and Piper
// Attention's key by the query's: tensors that do not match are refused here too, where a program can call
// the op itself.  Returns the device.
c10::Device checked_device(Operator op, const at::Tensor& q, const at::Tensor& k, const at::Tensor& v) {
  TORCH_CHECK(q.dim() == 4 && k.dim() == 4 && v.dim() == 4,
              "piper_kernels: tensors must have shape [batch, heads, sequence, head_dim]");
  TORCH_CHECK(k.device() == q.device() && v.device() == q.device(),
              "piper_kernels: query, key and value must share a device");
  // SageAttention2++'s prep reads no query: that has a type of its own, which is the output's
  TORCH_CHECK(v.scalar_type() == k.scalar_type() && (op == kSage || k.scalar_type() == q.scalar_type()),
              "piper_kernels: query, key and value must share a dtype");
  TORCH_CHECK(k.sizes() == v.sizes() && k.size(0) == q.size(0) && k.size(1) == q.size(1) && k.size(3) == q.size(3),
              "piper_kernels: batch, heads and head_dim must agree and key and value lengths match, got ", q.sizes(), ", ",
              k.sizes(), " and ", v.sizes());
  return q.device();
}

// What both operators' calls share: inputs, shape, output, stream.
struct Call {
  c10::OptionalDeviceGuard guard;
  at::Tensor query, key, value, output;
  piper_shape shape;
  int32_t dtype;
  c10::Stream stream;
  void* handle;

  Call(Operator op, const at::Tensor& q, const at::Tensor& k, const at::Tensor& v)
      : guard(checked_device(op, q, k, v)),
        query(native_input(q)),
        key(native_input(k)),
        value(native_input(v)),
        output(at::empty(q.sizes(), q.options().memory_format(at::MemoryFormat::Contiguous))),
        shape{q.size(0), q.size(1), q.size(2), k.size(2), q.size(3)},
        dtype(dtype_code(q)),
        stream(c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(q.device().index())),
        handle(static_cast<hipStream_t>(c10::hip::HIPStreamMasqueradingAsCUDA(stream))) {}

  at::Tensor workspace(const Arena& arena) const { return at::empty({arena.size}, query.options().dtype(at::kByte)); }

  // the caching allocator must not hand the inputs to another stream before this one has read them
  void keep_inputs() const {
    query.record_stream(stream);
    key.record_stream(stream);
    value.record_stream(stream);
  }
};

at::Tensor piper_attention(const at::Tensor& query, const at::Tensor& key, const at::Tensor& value, double scale,
                           bool is_causal) {
  Call call(kPiper, query, key, value);
  piper_layout layout;
  check(piper_prepared_layout(&call.shape, &layout), "piper_prepared_layout");  // refuses bad shapes
  const int32_t plan = plan_for(kPiper, call.shape, is_causal);
  int64_t attention_bytes = 0;
  check(piper_attention_workspace_bytes(&call.shape, plan, &attention_bytes), "piper_attention_workspace_bytes");

  Arena arena;
  const int64_t key_scale = arena.take(layout.key_scale_bytes);
  const int64_t value_scale = arena.take(layout.value_scale_bytes);
  const int64_t key_mean = arena.take(layout.mean_bytes);
  const int64_t value_mean = arena.take(layout.mean_bytes);
  const int64_t kv_tiles = arena.take(layout.kv_tiles_bytes);
  const int64_t prep = arena.take(layout.workspace_bytes);
  const int64_t attention = arena.take(attention_bytes);
  const at::Tensor memory = call.workspace(arena);
  char* base = static_cast<char*>(memory.mutable_data_ptr());
  const auto floats = [&](int64_t offset) { return reinterpret_cast<float*>(base + offset); };

  piper_prepare_args p{};
  p.abi_version = PIPER_ABI_VERSION;
  p.dtype = call.dtype;
  p.is_causal = is_causal;
  p.flags = PIPER_PREPARE_SKIP_QUERY | PIPER_PREPARE_QK_PER_THREAD;
  p.shape = call.shape;
  p.query = tensor_arg(call.query);
  p.key = tensor_arg(call.key);
  p.value = tensor_arg(call.value);
  p.prepared.key_scale = floats(key_scale);
  p.prepared.value_scale = floats(value_scale);
  p.prepared.key_mean = floats(key_mean);
  p.prepared.value_mean = floats(value_mean);
  p.prepared.kv_tiles = base + kv_tiles;
  p.workspace = base + prep;
  p.workspace_bytes = layout.workspace_bytes;
  check(piper_prepare(&p, call.handle), "piper_prepare");

  piper_attention_fused_args a{};
  a.abi_version = PIPER_ABI_VERSION;
  a.dtype = call.dtype;
  a.output_dtype = call.dtype;
  a.is_causal = is_causal;
  a.plan = plan;
  a.scale = static_cast<float>(scale);
  a.flags = PIPER_ATTENTION_QK_PER_THREAD;
  a.shape = call.shape;
  a.query = p.query;
  a.prepared = p.prepared;
  a.output = call.output.mutable_data_ptr();
  a.workspace = attention_bytes > 0 ? base + attention : nullptr;
  a.workspace_bytes = attention_bytes;
  check(piper_attention_forward_balanced(&a, call.handle), "piper_attention_forward_balanced");
  call.keep_inputs();
  return call.output;
}

at::Tensor sage_attention_2pp(const at::Tensor& query, const at::Tensor& key, const at::Tensor& value, double scale,
                              bool is_causal) {
  Call call(kSage, query, key, value);
  piper_sage_layout layout;
  check(piper_sage_prepared_layout(&call.shape, &layout), "piper_sage_prepared_layout");  // refuses bad shapes
  const int32_t plan = plan_for(kSage, call.shape, is_causal);

  Arena arena;
  const int64_t key_scale = arena.take(layout.key_scale_bytes);
  const int64_t key_mean = arena.take(layout.mean_bytes);
  const int64_t value_scale = arena.take(layout.mean_bytes);
  const int64_t kv_tiles = arena.take(layout.kv_tiles_bytes);
  const int64_t prep = arena.take(layout.workspace_bytes);
  const at::Tensor memory = call.workspace(arena);
  char* base = static_cast<char*>(memory.mutable_data_ptr());

  piper_sage_prepare_args p{};
  p.abi_version = PIPER_ABI_VERSION;
  p.dtype = dtype_code(key);
  p.flags = PIPER_PREPARE_QK_PER_THREAD;
  p.shape = call.shape;
  p.key = tensor_arg(call.key);
  p.value = tensor_arg(call.value);
  p.prepared.key_scale = reinterpret_cast<float*>(base + key_scale);
  p.prepared.key_mean = reinterpret_cast<float*>(base + key_mean);
  p.prepared.value_scale = reinterpret_cast<float*>(base + value_scale);
  p.prepared.kv_tiles = base + kv_tiles;
  p.workspace = base + prep;
  p.workspace_bytes = layout.workspace_bytes;
  check(piper_sage_prepare(&p, call.handle), "piper_sage_prepare");

  piper_sage_attention_args a{};
  a.abi_version = PIPER_ABI_VERSION;
  a.dtype = call.dtype;
  a.output_dtype = call.dtype;
  a.is_causal = is_causal;
  a.plan = plan;
  a.scale = static_cast<float>(scale);
  a.flags = PIPER_ATTENTION_QK_PER_THREAD;
  a.shape = call.shape;
  a.query = tensor_arg(call.query);
  a.prepared = p.prepared;
  a.output = call.output.mutable_data_ptr();
  check(piper_sage_attention_forward_balanced(&a, call.handle), "piper_sage_attention_forward_balanced");
  call.keep_inputs();
  return call.output;
}

}  // namespace

// What went wrong in the plan source: its text joins the error that the call raises.
extern "C" __attribute__((visibility("default"))) void piper_torch_plan_error(const char* text) {
  try {
    g_plan_error = text != nullptr ? text : "";
  } catch (const std::exception&) {  // out of memory: the call's error goes without the text
  }
}

// Sets the function that chooses launch plans, forgets the plans chosen so far and registers the kernels with
// torch (once; only here, so that no thread's call finds kernels without a plan source).  Returns NULL, or
// what went wrong.
extern "C" __attribute__((visibility("default"))) const char* piper_torch_set_plan_source(PlanSource source) {
  static thread_local std::string error;
  try {
    std::lock_guard<std::mutex> lock(g_plans_mutex);
    g_plan_source.store(source);
    g_plans.clear();
    static torch::Library* kernels = nullptr;  // registered until the process ends
    if (kernels == nullptr) {
      auto library = std::make_unique<torch::Library>(torch::Library::IMPL, "piper_kernels", c10::DispatchKey::CUDA,
                                                      __FILE__, __LINE__);
      library->impl("piper_attention", &piper_attention);
      library->impl("sage_attention_2pp", &sage_attention_2pp);
      kernels = library.release();
    }
  } catch (const std::exception& e) {
    error = e.what();
    return error.c_str();
  }
  return nullptr;
}
