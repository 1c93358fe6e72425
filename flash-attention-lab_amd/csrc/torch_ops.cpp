// The attention and decode ops as torch's dispatcher sees them, over the C ABI of
// include/flash_lab_hip.h (the reference registers its ops the same way, csrc/bindings.cpp:7-42).
//
// Each op checks its tensors (csrc/common/attn_host.h:18-57, csrc/decode/decode_host.h:18-53 of the
// reference), allocates the outputs and the workspace with torch's caching allocator on the inputs'
// device, and calls the library on the current stream. Nothing here synchronizes or reads seq_lens,
// so the ops can be captured in a HIP graph.
//
// Native because the call is what bounds a short decode: the same steps in Python, with the ctypes
// structures and the dispatcher's Python kernels, took 20 us for a decode of 9 us on the GPU.
//
// The library's functions are bound by address (fl_torch_bind), so that this file links against torch
// only and serves whichever build of the kernels was loaded.
#include <ATen/ATen.h>
#include <ATen/hip/HIPContext.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <c10/core/DeviceGuard.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/library.h>

#include <string>
#include <tuple>

#include "flash_lab_hip.h"

namespace {

using at::Tensor;
using Pair = std::tuple<Tensor, Tensor>;

struct Library {
  decltype(&fl_attention_plan) attention_plan;
  decltype(&fl_attention_fwd_split) attention_fwd_split;
  decltype(&fl_decode_plan) decode_plan;
  decltype(&fl_decode_schedule) decode_schedule;
  decltype(&fl_decode) decode;
  decltype(&fl_decode_balanced) decode_balanced;
  decltype(&fl_last_error) last_error;
};
Library lib{};

void check(int rc) { TORCH_CHECK(rc == FL_OK, lib.last_error()); }

const char* dtype_name(const Tensor& x) {
  switch (x.scalar_type()) {
    case at::kBFloat16: return "torch.bfloat16";
    case at::kHalf: return "torch.float16";
    case at::kFloat: return "torch.float32";
    default: return c10::toString(x.scalar_type());
  }
}

int32_t dtype_code(const Tensor& x) {
  return x.scalar_type() == at::kBFloat16 ? FL_DTYPE_BF16 : x.scalar_type() == at::kHalf ? FL_DTYPE_F16 : FL_DTYPE_F32;
}

void check_cuda(const Tensor& x, const char* name) { TORCH_CHECK(x.is_cuda(), name, " must be a CUDA tensor"); }

void check_rows(const Tensor& x, const char* name) {
  TORCH_CHECK(x.stride(-1) == 1, name, " must be contiguous in its last dimension");
}

int32_t cu_count(const Tensor& x) {
  return at::cuda::getDeviceProperties(x.device().index())->multiProcessorCount;
}

fl_stream_t current_stream(const Tensor& x) {
  return c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(x.device().index()).stream();
}

// A size that the library's int32 fields hold.
int32_t size32(int64_t n) {
  TORCH_CHECK(n <= INT32_MAX, "tensor dimension ", n, " is too large");
  return static_cast<int32_t>(n);
}

Pair attention(const Tensor& q, const Tensor& k_in, const Tensor& v_in, bool causal, double softmax_scale) {
  check_cuda(q, "q");
  check_cuda(k_in, "k");
  check_cuda(v_in, "v");
  TORCH_CHECK(q.scalar_type() == at::kBFloat16 || q.scalar_type() == at::kHalf,
              "attention_mma_pipelined takes bf16 or fp16");
  TORCH_CHECK(k_in.scalar_type() == q.scalar_type() && v_in.scalar_type() == q.scalar_type(),
              "k and v must have dtype ", dtype_name(q));
  TORCH_CHECK(q.dim() == 4 && k_in.dim() == 4 && v_in.dim() == 4, "q, k, v must be [B, S, H, D]");
  TORCH_CHECK(k_in.sizes() == v_in.sizes(), "k and v must have the same shape");
  TORCH_CHECK(q.size(0) == k_in.size(0) && q.size(3) == k_in.size(3),
              "q and k must agree on batch size and head_dim");
  TORCH_CHECK(q.device() == k_in.device() && q.device() == v_in.device(), "q, k, v on different devices");
  check_rows(q, "q");
  check_rows(k_in, "k");
  check_rows(v_in, "v");
  // The kernels need non-overlapping K and V rows (sequence stride >= head_dim); broadcast or
  // overlapping views, which the reference also accepts, are passed as contiguous copies.
  auto rows = [&](const Tensor& x) { return x.size(1) > 1 && x.stride(1) < x.size(3) ? x.contiguous() : x; };
  const Tensor k = rows(k_in);
  const Tensor v = rows(v_in);
  const c10::DeviceGuard guard(q.device());
  Tensor o = at::empty(q.sizes(), q.options().memory_format(at::MemoryFormat::Contiguous));
  Tensor lse = at::empty({q.size(0), q.size(2), q.size(1)}, q.options().dtype(at::kFloat));

  fl_attn_params p{};
  p.q = q.const_data_ptr();
  p.k = k.const_data_ptr();
  p.v = v.const_data_ptr();
  p.o = o.data_ptr();
  p.lse = lse.data_ptr<float>();
  p.q_batch_stride = q.stride(0), p.q_seq_stride = q.stride(1), p.q_head_stride = q.stride(2);
  p.k_batch_stride = k.stride(0), p.k_seq_stride = k.stride(1), p.k_head_stride = k.stride(2);
  p.v_batch_stride = v.stride(0), p.v_seq_stride = v.stride(1), p.v_head_stride = v.stride(2);
  p.o_batch_stride = o.stride(0), p.o_seq_stride = o.stride(1), p.o_head_stride = o.stride(2);
  p.batch = size32(q.size(0));
  p.seqlen_q = size32(q.size(1));
  p.seqlen_k = size32(k.size(1));
  p.heads = size32(q.size(2));
  p.heads_kv = size32(k.size(2));
  p.head_dim = size32(q.size(3));
  p.causal = causal;
  p.dtype = dtype_code(q);
  p.softmax_scale = softmax_scale;
  const fl_stream_t stream = current_stream(q);
  const int32_t cus = cu_count(q);
  const int rc = lib.attention_fwd_split(&p, 0, cus, nullptr, 0, stream);
  if (rc != FL_ERR_WORKSPACE) {
    check(rc);
    return {o, lse};
  }
  int32_t splits = 0;
  size_t bytes = 0;
  check(lib.attention_plan(&p, 0, cus, &splits, &bytes));
  Tensor workspace = at::empty({static_cast<int64_t>(bytes / sizeof(float))}, lse.options());
  check(lib.attention_fwd_split(&p, splits, cus, workspace.data_ptr<float>(), bytes, stream));
  return {o, lse};
}

Pair decode(const Tensor& q, const Tensor& k_cache, const Tensor& v_cache, const Tensor& seq_lens,
            const Tensor* block_tables, double softmax_scale, int64_t num_splits, bool allow_splits) {
  check_cuda(q, "q");
  check_cuda(k_cache, "k_cache");
  check_cuda(v_cache, "v_cache");
  check_cuda(seq_lens, "seq_lens");
  TORCH_CHECK(q.scalar_type() == at::kBFloat16 || q.scalar_type() == at::kHalf || q.scalar_type() == at::kFloat,
              "decode takes bf16, fp16, or fp32");
  TORCH_CHECK(k_cache.scalar_type() == q.scalar_type() && v_cache.scalar_type() == q.scalar_type(),
              "k_cache and v_cache must have dtype ", dtype_name(q));
  TORCH_CHECK(seq_lens.scalar_type() == at::kInt, "seq_lens must have dtype int32");
  TORCH_CHECK(q.dim() == 3 && k_cache.dim() == 4, "q must be [B, H, D], caches [B, S_max, H_kv, D]");
  TORCH_CHECK(k_cache.sizes() == v_cache.sizes(), "k_cache and v_cache must have the same shape");
  if (block_tables == nullptr) {
    TORCH_CHECK(k_cache.size(0) == q.size(0) && k_cache.size(3) == q.size(2),
                "q and the caches must agree on batch size and head_dim");
  } else {
    check_cuda(*block_tables, "block_tables");
    TORCH_CHECK(block_tables->scalar_type() == at::kInt, "block_tables must have dtype int32");
    TORCH_CHECK(block_tables->dim() == 2 && block_tables->size(0) == q.size(0) && block_tables->size(1) >= 1 &&
                    block_tables->stride(1) == 1,
                "block_tables must be [B, max_blocks] with unit stride in its last dimension");
    TORCH_CHECK(k_cache.size(3) == q.size(2), "q and the caches must agree on head_dim");
    TORCH_CHECK(block_tables->size(1) * k_cache.size(1) <= INT32_MAX,
                "paged cache too long (max_blocks * page_size must fit in int32)");
  }
  TORCH_CHECK(seq_lens.dim() == 1 && seq_lens.size(0) == q.size(0), "seq_lens must be [B]");
  TORCH_CHECK(seq_lens.is_contiguous(), "seq_lens must be contiguous");
  check_rows(q, "q");
  check_rows(k_cache, "k_cache");
  check_rows(v_cache, "v_cache");
  TORCH_CHECK(0 <= num_splits && num_splits <= 128, "num_splits must be in [0, 128]");

  const c10::DeviceGuard guard(q.device());
  Tensor o = at::empty(q.sizes(), q.options().memory_format(at::MemoryFormat::Contiguous));
  Tensor lse = at::empty({q.size(0), q.size(1)}, q.options().dtype(at::kFloat));
  fl_decode_params p{};
  p.q = q.const_data_ptr();
  p.k_cache = k_cache.const_data_ptr();
  p.v_cache = v_cache.const_data_ptr();
  p.o = o.data_ptr();
  p.lse = lse.data_ptr<float>();
  p.seq_lens = seq_lens.const_data_ptr<int32_t>();
  p.q_batch_stride = q.stride(0), p.q_head_stride = q.stride(1);
  p.k_batch_stride = k_cache.stride(0), p.k_seq_stride = k_cache.stride(1), p.k_head_stride = k_cache.stride(2);
  p.v_batch_stride = v_cache.stride(0), p.v_seq_stride = v_cache.stride(1), p.v_head_stride = v_cache.stride(2);
  p.o_batch_stride = o.stride(0), p.o_head_stride = o.stride(1);
  p.batch = size32(q.size(0));
  p.heads = size32(q.size(1));
  p.heads_kv = size32(k_cache.size(2));
  p.head_dim = size32(q.size(2));
  p.max_seqlen = size32(k_cache.size(1));
  p.num_splits = 1;
  p.dtype = dtype_code(q);
  p.softmax_scale = softmax_scale;
  if (block_tables != nullptr) {
    // [num_blocks, page_size, H_kv, D] caches: the batch strides are block strides.
    p.max_seqlen = size32(block_tables->size(1) * k_cache.size(1));
    p.block_tables = block_tables->const_data_ptr<int32_t>();
    p.block_tables_stride = block_tables->stride(0);
    p.page_size = size32(k_cache.size(1));
    p.num_blocks = size32(k_cache.size(0));
  }
  int32_t splits = 0;
  int32_t workgroups = 0;
  if (allow_splits && num_splits == 0) {
    check(lib.decode_schedule(&p, cu_count(q), &splits, &workgroups, &p.workspace_bytes));
  } else {
    check(lib.decode_plan(&p, static_cast<int32_t>(num_splits), allow_splits, cu_count(q), &splits, &p.workspace_bytes));
  }
  p.num_splits = splits;
  Tensor workspace;
  if (p.workspace_bytes > 0) {
    workspace = at::empty({static_cast<int64_t>(p.workspace_bytes / sizeof(float))}, lse.options());
    p.workspace = workspace.data_ptr<float>();
  }
  const fl_stream_t stream = current_stream(q);
  check(workgroups > 0 ? lib.decode_balanced(&p, workgroups, stream) : lib.decode(&p, stream));
  return {o, lse};
}

template <bool kSplits>
Pair decode_op(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& seq_lens, double scale,
               int64_t num_splits) {
  return decode(q, k, v, seq_lens, nullptr, scale, num_splits, kSplits);
}

template <bool kSplits>
Pair paged_decode_op(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& seq_lens,
                     const Tensor& block_tables, double scale, int64_t num_splits) {
  return decode(q, k, v, seq_lens, &block_tables, scale, num_splits, kSplits);
}

// The ops have no gradient. With inputs that require one, the outputs are part of the graph and a
// backward through them raises; otherwise the call goes straight on below autograd.
template <typename... Args>
struct NoGradient {
  using Op = c10::TypedOperatorHandle<Pair(Args...)>;
  struct Node : torch::autograd::Function<Node> {
    static torch::autograd::variable_list forward(torch::autograd::AutogradContext* ctx, const Op& op,
                                                  const std::string& name, Args... args) {
      ctx->saved_data["op"] = name;
      at::AutoDispatchBelowADInplaceOrView below;
      auto [o, lse] = op.call(args...);
      return {o, lse};
    }
    static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx,
                                                   torch::autograd::variable_list) {
      TORCH_CHECK(false, "Trying to backward through flash_lab.", ctx->saved_data["op"].toStringRef(),
                  ".default but no autograd formula was registered. Please use register_autograd to add one.");
    }
  };
  static bool requires_grad(const Tensor& x) { return x.requires_grad(); }
  template <typename T>
  static bool requires_grad(const T&) {
    return false;
  }
  static Pair call(const char* name, const Op& op, Args... args) {
    if (at::GradMode::is_enabled() && (requires_grad(args) || ...)) {
      auto outputs = Node::apply(op, std::string(name), args...);
      return {outputs[0], outputs[1]};
    }
    at::AutoDispatchBelowADInplaceOrView below;
    return op.call(args...);
  }
};

using Prefill = NoGradient<const Tensor&, const Tensor&, const Tensor&, bool, double>;
using Decode = NoGradient<const Tensor&, const Tensor&, const Tensor&, const Tensor&, double, int64_t>;
using PagedDecode =
    NoGradient<const Tensor&, const Tensor&, const Tensor&, const Tensor&, const Tensor&, double, int64_t>;

#define FL_AUTOGRAD(kind, op_name, params, args)                                                        \
  Pair op_name##_autograd params {                                                                       \
    static const auto op = c10::Dispatcher::singleton().findSchemaOrThrow("flash_lab::" #op_name, "")    \
                               .typed<Pair params>();                                                    \
    return kind::call args;                                                                              \
  }
FL_AUTOGRAD(Prefill, attention_mma_pipelined,
            (const Tensor& q, const Tensor& k, const Tensor& v, bool causal, double scale),
            ("attention_mma_pipelined", op, q, k, v, causal, scale))
FL_AUTOGRAD(Prefill, attention_mma, (const Tensor& q, const Tensor& k, const Tensor& v, bool causal, double scale),
            ("attention_mma", op, q, k, v, causal, scale))
#define FL_DECODE_AUTOGRAD(name)                                                                         \
  FL_AUTOGRAD(Decode, name,                                                                              \
              (const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& lens, double scale, int64_t n), \
              (#name, op, q, k, v, lens, scale, n))
#define FL_PAGED_AUTOGRAD(name)                                                                          \
  FL_AUTOGRAD(PagedDecode, name,                                                                         \
              (const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& lens, const Tensor& tables, \
               double scale, int64_t n),                                                                 \
              (#name, op, q, k, v, lens, tables, scale, n))
FL_DECODE_AUTOGRAD(decode_splitkv)
FL_DECODE_AUTOGRAD(decode_inplace)
FL_PAGED_AUTOGRAD(decode_splitkv_paged)
FL_PAGED_AUTOGRAD(decode_inplace_paged)

}  // namespace

// The reference's schemas, verbatim (csrc/bindings.cpp:9-41); the paged forms, which the reference
// lacks (its kernels reject paged caches), take the block tables after seq_lens.
TORCH_LIBRARY_FRAGMENT(flash_lab, m) {
  const char* prefill = "(Tensor q, Tensor k, Tensor v, bool causal, float softmax_scale) -> (Tensor, Tensor)";
  const char* decode = "(Tensor q, Tensor k_cache, Tensor v_cache, Tensor seq_lens, float softmax_scale,"
                       " int num_splits) -> (Tensor, Tensor)";
  const char* paged = "(Tensor q, Tensor k_cache, Tensor v_cache, Tensor seq_lens, Tensor block_tables,"
                      " float softmax_scale, int num_splits) -> (Tensor, Tensor)";
  auto def = [&](const char* name, const char* schema) {
    m.def(torch::schema((std::string(name) + schema).c_str()), {at::Tag::pt2_compliant_tag});
  };
  def("attention_mma_pipelined", prefill);
  def("attention_mma", prefill);
  def("decode_splitkv", decode);
  def("decode_inplace", decode);
  def("decode_splitkv_paged", paged);
  def("decode_inplace_paged", paged);
}

TORCH_LIBRARY_IMPL(flash_lab, CUDA, m) {
  m.impl("attention_mma_pipelined", &attention);
  m.impl("attention_mma", &attention);
  m.impl("decode_splitkv", &decode_op<true>);
  m.impl("decode_inplace", &decode_op<false>);
  m.impl("decode_splitkv_paged", &paged_decode_op<true>);
  m.impl("decode_inplace_paged", &paged_decode_op<false>);
}

TORCH_LIBRARY_IMPL(flash_lab, Autograd, m) {
  m.impl("attention_mma_pipelined", &attention_mma_pipelined_autograd);
  m.impl("attention_mma", &attention_mma_autograd);
  m.impl("decode_splitkv", &decode_splitkv_autograd);
  m.impl("decode_inplace", &decode_inplace_autograd);
  m.impl("decode_splitkv_paged", &decode_splitkv_paged_autograd);
  m.impl("decode_inplace_paged", &decode_inplace_paged_autograd);
}

// The addresses of the library's functions, in this order; once, before the first call of an op.
extern "C" void fl_torch_bind(void* attention_plan, void* attention_fwd_split, void* decode_plan,
                              void* decode_schedule, void* decode, void* decode_balanced, void* last_error) {
  lib.attention_plan = reinterpret_cast<decltype(lib.attention_plan)>(attention_plan);
  lib.attention_fwd_split = reinterpret_cast<decltype(lib.attention_fwd_split)>(attention_fwd_split);
  lib.decode_plan = reinterpret_cast<decltype(lib.decode_plan)>(decode_plan);
  lib.decode_schedule = reinterpret_cast<decltype(lib.decode_schedule)>(decode_schedule);
  lib.decode = reinterpret_cast<decltype(lib.decode)>(decode);
  lib.decode_balanced = reinterpret_cast<decltype(lib.decode_balanced)>(decode_balanced);
  lib.last_error = reinterpret_cast<decltype(lib.last_error)>(last_error);
}
