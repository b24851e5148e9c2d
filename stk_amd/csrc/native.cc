// The Python boundary in native code: what stk_amd/backend/hip_kernels.py checks, allocates and launches, as one call
// per operation on torch tensors.  The checks, the errors they raise and the launches are those of the C ABI
// (include/stk_amd.h); what this saves is the host time of a launch.  Through ctypes, with the checks in Python, a call
// took 10 - 14 us on the host, more than most kernels of a small problem take on the GPU; here it takes 3 - 5 us.
//
// Everything - copies of operands, allocations, launches - happens on torch's current stream of the tensors' device.  No
// state is kept between calls but one pinned word per host thread and device (Mailbox).
#include <torch/extension.h>

#include <c10/hip/HIPStream.h>
#include <hip/hip_runtime_api.h>

#include <optional>
#include <string>
#include <tuple>
#include <vector>

#include "../../include/stk_amd.h"

namespace {

using at::Tensor;
using OptTensor = std::optional<Tensor>;

// ------------------------------------------------------------------------------------------------ errors
// (the functions run without the interpreter's lock)
[[noreturn]] void raise(PyObject* type, const std::string& text) {
  py::gil_scoped_acquire gil;
  PyErr_SetString(type, text.c_str());
  throw py::error_already_set();
}
void require(bool ok, const char* text) {
  if (!ok) raise(PyExc_AssertionError, text);
}
// The exception that the reference raises in the same situation.
void check(int status) {
  if (status == STK_OK) return;
  raise(status == STK_ERR_DIMS ? PyExc_AssertionError : status == STK_ERR_UNSUPPORTED ? PyExc_NotImplementedError : PyExc_RuntimeError,
        stk_last_error());
}
void need_gpu(const Tensor& t) {
  if (!t.is_cuda()) raise(PyExc_RuntimeError, "stk_amd: this operation runs on a ROCm GPU only; got a tensor on " + t.device().str());
}

// ------------------------------------------------------------------------------------------------ operands
int value_dtype(const Tensor& t) {
  switch (t.scalar_type()) {
    case at::kHalf: return STK_F16;
    case at::kBFloat16: return STK_BF16;
    case at::kFloat: return STK_F32;
    default:
      raise(PyExc_NotImplementedError, std::string("stk_amd: products need float16, bfloat16 or float32 values, got ") + c10::toString(t.scalar_type()));
  }
}
int index_dtype(at::ScalarType t) {
  if (t == at::kShort) return STK_I16;
  if (t == at::kInt) return STK_I32;
  raise(PyExc_NotImplementedError, std::string("stk_amd: indices must be int16 or int32, got ") + c10::toString(t));
}
// Index tensors may arrive as strided views (stk/ops/matrix_ops.py:73-75).
Tensor index(const Tensor& t) {
  index_dtype(t.scalar_type());
  return t.contiguous();
}
Tensor offsets32(const Tensor& t) {
  if (t.scalar_type() != at::kInt) raise(PyExc_NotImplementedError, std::string("stk_amd: offsets must be int32, got ") + c10::toString(t.scalar_type()));
  return t.contiguous();
}
bool aligned(const Tensor& t) { return (reinterpret_cast<uintptr_t>(t.const_data_ptr()) & 15u) == 0; }
// A 2-D operand the kernels can read in place: unit stride in one dimension, the other stride a multiple of 8
// elements, 16-byte aligned base.  Anything else is copied to row-major first.
Tensor dense_operand(const Tensor& x) {
  require(x.dim() == 2, "dense operands have two dimensions");
  const int64_t s0 = x.stride(0), s1 = x.stride(1);
  if (((s1 == 1 && s0 % 8 == 0) || (s0 == 1 && s1 % 8 == 0 && x.size(0) > 1)) && aligned(x)) return x;
  Tensor c = x.contiguous();
  if (!aligned(c) || c.stride(0) % 8) raise(PyExc_NotImplementedError, "stk_amd: dense operands need a row length divisible by 8");
  return c;
}
void matmul_dims(int64_t m, int64_t k, int64_t n, int64_t b) {
  // stk/backend/triton_kernels.py:15-19 with BLOCK_M = BLOCK_N = blocking, BLOCK_K = 32
  const auto test = [](int64_t v, int64_t by) {
    if (by == 0 || v % by)
      raise(PyExc_AssertionError, "incompatible dimensions: tensor has dim with length: " + std::to_string(v) + ", which must be divisible by " + std::to_string(by));
  };
  test(m, b);
  test(k, 32);
  test(n, b);
}
template <class T>
T* ptr(const Tensor& t) { return static_cast<T*>(const_cast<void*>(t.const_data_ptr())); }
template <class T>
T* ptr(const OptTensor& t) { return t ? ptr<T>(*t) : nullptr; }

// The stream a call launches on.
hipStream_t stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

// ------------------------------------------------------------------------------------------------ products
// The sparse operand's arrays as the launches take them.
struct Meta {
  Tensor offsets, ci, offsets_t, cit, bot;
  int idx;
  Meta(const Tensor& offsets_, const Tensor& ci_, const Tensor& offsets_t_, const Tensor& cit_, const Tensor& bot_)
      : offsets(offsets32(offsets_)), ci(index(ci_)), offsets_t(offsets32(offsets_t_)), cit(index(cit_)), bot(offsets32(bot_)),
        idx(index_dtype(ci.scalar_type())) {}
};
#define META_ARGS const Tensor &offsets, const Tensor &column_indices, const Tensor &offsets_t, const Tensor &column_indices_t, const Tensor &block_offsets_t
#define META_PTRS(m) ptr<int32_t>(m.offsets), ptr<void>(m.ci), ptr<int32_t>(m.offsets_t), ptr<void>(m.cit), ptr<int32_t>(m.bot)

void sdd(const Tensor& lhs_, const Tensor& rhs_, const Tensor& out, const OptTensor& offsets, const Tensor& row_indices, const Tensor& column_indices,
         const OptTensor& plan, int activation, const OptTensor& multiplier, const OptTensor& block_order, const OptTensor& sums) {
  need_gpu(lhs_), need_gpu(rhs_), need_gpu(out);
  require(lhs_.dim() == 2 && rhs_.dim() == 2 && lhs_.size(1) == rhs_.size(0), "incompatible dimensions");
  const int64_t m = lhs_.size(0), k = lhs_.size(1), n = rhs_.size(1), b = out.size(-1), nnz = row_indices.numel();
  matmul_dims(m, k, n, b);
  require(out.is_contiguous(), "out must be contiguous");
  const auto like_out = [&](const OptTensor& t, const char* text) {
    if (!t) return;
    need_gpu(*t);
    require(t->sizes() == out.sizes() && t->scalar_type() == out.scalar_type() && t->is_contiguous(), text);
  };
  like_out(multiplier, "the multiplier's values must be laid out like out");
  like_out(sums, "sums must be laid out like out");
  require(!sums || sums->const_data_ptr() != out.const_data_ptr(), "sums need an array of their own");
  if (nnz == 0) return;
  const c10::DeviceGuard guard(out.device());
  const Tensor lhs = dense_operand(lhs_), rhs = dense_operand(rhs_);
  require(lhs.scalar_type() == rhs.scalar_type() && lhs.scalar_type() == out.scalar_type(), "operands and out must have one dtype");
  const Tensor ri = index(row_indices), ci = index(column_indices);
  require(ri.scalar_type() == ci.scalar_type(), "row and column indices must have one dtype");
  OptTensor order;
  if (block_order) {
    require(block_order->scalar_type() == at::kInt && block_order->numel() == nnz, "block_order must be an int32 permutation of the blocks");
    order = block_order->contiguous();
  }
  OptTensor offs;
  if (plan) offs = offsets32(*offsets);
  check(stk_sdd_fused_sums(ptr<void>(lhs), lhs.stride(0), lhs.stride(1), ptr<void>(rhs), rhs.stride(0), rhs.stride(1), m, k, n, ptr<void>(out),
                           ptr<int32_t>(offs), ptr<void>(ri), ptr<void>(ci), ptr<int32_t>(order), nnz, (int)b, value_dtype(out),
                           index_dtype(ri.scalar_type()), ptr<uint8_t>(plan), activation, ptr<void>(multiplier), ptr<void>(sums), stream_of(out)));
}

// The status of the launch: the caller owns the workspace, whose state depends on it.  (Operands that are refused raise.)
int dsd(int64_t m, int64_t k, const Tensor& data, META_ARGS, bool transpose_a, const Tensor& rhs_, const Tensor& out, const OptTensor& plan,
        const OptTensor& workspace) {
  need_gpu(data), need_gpu(rhs_), need_gpu(out);
  require(rhs_.dim() == 2 && k == rhs_.size(0), "incompatible dimensions");
  const int64_t n = rhs_.size(1), b = data.size(-1);
  matmul_dims(m, k, n, b);
  const c10::DeviceGuard guard(out.device());
  const Tensor rhs = dense_operand(rhs_);
  require(data.is_contiguous() && out.stride(1) == 1, "the sparse values must be contiguous and out row-major");
  require(data.scalar_type() == rhs.scalar_type() && data.scalar_type() == out.scalar_type(), "operands and out must have one dtype");
  const Meta s(offsets, column_indices, offsets_t, column_indices_t, block_offsets_t);
  return stk_dsd(m, k, n, ptr<void>(data), META_PTRS(s), transpose_a, ptr<void>(rhs), rhs.stride(0), rhs.stride(1), ptr<void>(out), out.stride(0),
                 data.size(0), (int)b, value_dtype(out), s.idx, ptr<uint8_t>(plan), ptr<void>(workspace), workspace ? workspace->numel() : 0,
                 stream_of(out));
}

void dds(const Tensor& lhs_, int64_t k, int64_t n, const Tensor& data, META_ARGS, bool transpose_b, const Tensor& out, const OptTensor& plan) {
  need_gpu(data), need_gpu(lhs_), need_gpu(out);
  require(lhs_.dim() == 2 && lhs_.size(1) == k, "incompatible dimensions");
  const int64_t m = lhs_.size(0), b = data.size(-1);
  matmul_dims(m, k, n, b);
  const c10::DeviceGuard guard(out.device());
  const Tensor lhs = dense_operand(lhs_);
  require(data.is_contiguous() && out.stride(1) == 1, "the sparse values must be contiguous and out row-major");
  require(data.scalar_type() == lhs.scalar_type() && data.scalar_type() == out.scalar_type(), "operands and out must have one dtype");
  const Meta s(offsets, column_indices, offsets_t, column_indices_t, block_offsets_t);
  check(stk_dds(m, k, n, ptr<void>(lhs), lhs.stride(0), lhs.stride(1), ptr<void>(data), META_PTRS(s), transpose_b, ptr<void>(out), out.stride(0),
                data.size(0), (int)b, value_dtype(out), s.idx, ptr<uint8_t>(plan), stream_of(out)));
}

void dsd_dds(int64_t m, int64_t k, const Tensor& data, META_ARGS, const Tensor& rhs_, const Tensor& out_dsd, const Tensor& lhs_, const Tensor& out_dds,
             const OptTensor& plan) {
  need_gpu(data), need_gpu(rhs_), need_gpu(lhs_), need_gpu(out_dsd), need_gpu(out_dds);
  require(rhs_.dim() == 2 && lhs_.dim() == 2 && rhs_.size(0) == k && lhs_.size(1) == m, "incompatible dimensions");
  const int64_t b = data.size(-1);
  matmul_dims(m, k, rhs_.size(1), b);
  matmul_dims(lhs_.size(0), m, k, b);
  const c10::DeviceGuard guard(data.device());
  const Tensor rhs = dense_operand(rhs_), lhs = dense_operand(lhs_);
  require(data.is_contiguous() && out_dsd.stride(1) == 1 && out_dds.stride(1) == 1, "the sparse values must be contiguous and the results row-major");
  const auto t = data.scalar_type();
  require(rhs.scalar_type() == t && lhs.scalar_type() == t && out_dsd.scalar_type() == t && out_dds.scalar_type() == t, "operands and results must have one dtype");
  const Meta s(offsets, column_indices, offsets_t, column_indices_t, block_offsets_t);
  check(stk_dsd_dds(m, k, ptr<void>(data), META_PTRS(s), rhs.size(1), ptr<void>(rhs), rhs.stride(0), rhs.stride(1), ptr<void>(out_dsd), out_dsd.stride(0),
                    lhs.size(0), ptr<void>(lhs), lhs.stride(0), lhs.stride(1), ptr<void>(out_dds), out_dds.stride(0), data.size(0), (int)b,
                    value_dtype(data), s.idx, ptr<uint8_t>(plan), stream_of(data)));
}

void dsd_dsd(int64_t m, int64_t k, const Tensor& data, META_ARGS, const Tensor& rhs_, const Tensor& out, const Tensor& rhs_t_, const Tensor& out_t,
             const OptTensor& plan) {
  need_gpu(data), need_gpu(rhs_), need_gpu(rhs_t_), need_gpu(out), need_gpu(out_t);
  require(rhs_.dim() == 2 && rhs_t_.dim() == 2 && rhs_.size(0) == k && rhs_t_.size(0) == m, "incompatible dimensions");
  const int64_t b = data.size(-1);
  matmul_dims(m, k, rhs_.size(1), b);
  matmul_dims(k, m, rhs_t_.size(1), b);
  const c10::DeviceGuard guard(data.device());
  const Tensor rhs = dense_operand(rhs_), rhs_t = dense_operand(rhs_t_);
  require(data.is_contiguous() && out.stride(1) == 1 && out_t.stride(1) == 1, "the sparse values must be contiguous and the results row-major");
  const auto t = data.scalar_type();
  require(rhs.scalar_type() == t && rhs_t.scalar_type() == t && out.scalar_type() == t && out_t.scalar_type() == t, "operands and results must have one dtype");
  const Meta s(offsets, column_indices, offsets_t, column_indices_t, block_offsets_t);
  check(stk_dsd_dsd(m, k, ptr<void>(data), META_PTRS(s), rhs.size(1), ptr<void>(rhs), rhs.stride(0), rhs.stride(1), ptr<void>(out), out.stride(0),
                    rhs_t.size(1), ptr<void>(rhs_t), rhs_t.stride(0), rhs_t.stride(1), ptr<void>(out_t), out_t.stride(0), data.size(0), (int)b,
                    value_dtype(data), s.idx, ptr<uint8_t>(plan), stream_of(data)));
}

void sdd_dsd(int64_t m, int64_t n, const Tensor& lhs_, const Tensor& rhs_sdd_, const Tensor& out_sdd, const Tensor& data, const Tensor& row_indices,
             META_ARGS, bool transpose_a, const Tensor& rhs_dsd_, const Tensor& out_dsd, const OptTensor& plan) {
  need_gpu(data), need_gpu(lhs_), need_gpu(rhs_sdd_), need_gpu(rhs_dsd_), need_gpu(out_sdd), need_gpu(out_dsd);
  const int64_t b = data.size(-1);
  require(lhs_.dim() == 2 && rhs_sdd_.dim() == 2 && rhs_dsd_.dim() == 2 && lhs_.size(0) == m && rhs_sdd_.size(1) == n && lhs_.size(1) == rhs_sdd_.size(0) &&
              rhs_dsd_.size(0) == (transpose_a ? m : n), "incompatible dimensions");
  matmul_dims(m, lhs_.size(1), n, b);
  matmul_dims(transpose_a ? n : m, rhs_dsd_.size(0), rhs_dsd_.size(1), b);
  const c10::DeviceGuard guard(data.device());
  const Tensor lhs = dense_operand(lhs_), rhs_sdd = dense_operand(rhs_sdd_), rhs_dsd = dense_operand(rhs_dsd_);
  require(data.is_contiguous() && out_sdd.is_contiguous() && out_sdd.sizes() == data.sizes() && out_dsd.stride(1) == 1,
          "the sparse values must be contiguous and the results laid out like them and row-major");
  const auto t = data.scalar_type();
  require(lhs.scalar_type() == t && rhs_sdd.scalar_type() == t && rhs_dsd.scalar_type() == t && out_sdd.scalar_type() == t && out_dsd.scalar_type() == t,
          "operands and results must have one dtype");
  const Tensor ri = index(row_indices);
  const Meta s(offsets, column_indices, offsets_t, column_indices_t, block_offsets_t);
  require(ri.scalar_type() == s.ci.scalar_type() && ri.scalar_type() == s.cit.scalar_type(), "the indices must have one dtype");
  check(stk_sdd_dsd(m, n, ptr<int32_t>(s.offsets), ptr<void>(ri), ptr<void>(s.ci), ptr<int32_t>(s.offsets_t), ptr<void>(s.cit), ptr<int32_t>(s.bot),
                    ptr<void>(lhs), lhs.stride(0), lhs.stride(1), ptr<void>(rhs_sdd), rhs_sdd.stride(0), rhs_sdd.stride(1), lhs.size(1), ptr<void>(out_sdd),
                    ptr<void>(data), transpose_a, rhs_dsd.size(1), ptr<void>(rhs_dsd), rhs_dsd.stride(0), rhs_dsd.stride(1), ptr<void>(out_dsd),
                    out_dsd.stride(0), data.size(0), (int)b, value_dtype(data), s.idx, ptr<uint8_t>(plan), stream_of(data)));
}

// ------------------------------------------------------------------------------------------------ plan, streams, workspaces
Tensor build_plan(const Tensor& offsets_, const Tensor& column_indices, const OptTensor& offsets_t_, const OptTensor& column_indices_t, int blocking) {
  need_gpu(offsets_), need_gpu(column_indices);
  const c10::DeviceGuard guard(offsets_.device());
  const Tensor offsets = offsets32(offsets_), ci = index(column_indices);
  OptTensor offsets_t, cit;
  if (offsets_t_ && column_indices_t) offsets_t = offsets32(*offsets_t_), cit = index(*column_indices_t);
  const int64_t rows = offsets.numel() - 1, cols = offsets_t ? offsets_t->numel() - 1 : 0, nnz = ci.numel();
  const int64_t bytes = (int64_t)stk_plan_bytes(rows, cols, nnz);
  Tensor plan = at::empty({bytes > 0 ? bytes : 1}, offsets.options().dtype(at::kByte));
  check(stk_build_plan(ptr<int32_t>(offsets), ptr<void>(ci), rows, ptr<int32_t>(offsets_t), ptr<void>(cit), cols, nnz, blocking,
                       index_dtype(ci.scalar_type()), ptr<uint8_t>(plan), (size_t)bytes, stream_of(offsets)));
  return plan;
}

uint64_t capture_id(int64_t stream) {
  uint64_t id = 0;
  check(stk_stream_capture_id(reinterpret_cast<stk_stream_t>(stream), &id));
  return id;
}

// What is launched on the stream `waiting` from now on starts after what has been launched on `first`.
void follow(int64_t waiting, int64_t first) {
  const auto test = [](hipError_t e) {
    if (e != hipSuccess) raise(PyExc_RuntimeError, std::string("stk_amd: ordering two streams: ") + hipGetErrorString(e));
  };
  hipEvent_t event;
  test(hipEventCreateWithFlags(&event, hipEventDisableTiming));
  hipError_t e = hipEventRecord(event, reinterpret_cast<hipStream_t>(first));
  if (e == hipSuccess) e = hipStreamWaitEvent(reinterpret_cast<hipStream_t>(waiting), event, 0);
  (void)hipEventDestroy(event);   // (released once it has been reached)
  test(e);
}

// A word of pinned host memory that a kernel writes a count into and the host polls: one per host thread and device,
// in use only until the call that took it returns.
struct Mailbox {
  volatile int32_t* word;
  explicit Mailbox(const at::Device& device) {
    static thread_local std::vector<Tensor> words;
    const size_t at = (size_t)device.index();
    if (words.size() <= at) words.resize(at + 1);
    if (!words[at].defined()) words[at] = at::empty({1}, at::TensorOptions().dtype(at::kInt).pinned_memory(true));
    word = ptr<int32_t>(words[at]);
    *word = -1;
  }
  // The count.  Polled for a while - a stream wait costs more than the kernels of a small problem - then waited for, which
  // also reports a launch that failed.
  int32_t receive(hipStream_t stream) const {
    for (int i = 0; i < 200000 && *word < 0; i++) __builtin_ia32_pause();
    if (*word < 0) {
      const hipError_t e = hipStreamSynchronize(stream);
      if (e != hipSuccess || *word < 0)
        raise(PyExc_RuntimeError, e != hipSuccess ? std::string("stk_amd: ") + hipGetErrorString(e) : "stk_amd: the count was not delivered");
    }
    return *word;
  }
};

// ------------------------------------------------------------------------------------------------ topology and formats
void row_indices(const Tensor& offsets_, const Tensor& out) {
  need_gpu(offsets_), need_gpu(out);
  require(out.is_contiguous(), "out must be contiguous");
  const c10::DeviceGuard guard(out.device());
  const Tensor offsets = offsets32(offsets_);
  check(stk_row_indices(ptr<int32_t>(offsets), offsets.numel() - 1, out.numel(), ptr<void>(out), index_dtype(out.scalar_type()), stream_of(out)));
}

std::tuple<Tensor, Tensor, Tensor> transpose_meta(int64_t block_cols, const Tensor& row_indices, const Tensor& column_indices) {
  need_gpu(row_indices), need_gpu(column_indices);
  const c10::DeviceGuard guard(column_indices.device());
  const Tensor ri = index(row_indices), ci = index(column_indices);
  require(ri.scalar_type() == ci.scalar_type(), "row and column indices must have one dtype");
  const int64_t nnz = ci.numel();
  Tensor cit = at::empty({nnz}, ri.options()), offsets_t = at::empty({block_cols + 1}, ri.options().dtype(at::kInt));
  Tensor bot = at::empty({nnz}, offsets_t.options());
  const size_t bytes = stk_transpose_meta_workspace_bytes(nnz);
  Tensor ws = at::empty({(int64_t)bytes}, ri.options().dtype(at::kByte));
  check(stk_transpose_meta(ptr<void>(ri), ptr<void>(ci), nnz, block_cols, index_dtype(ci.scalar_type()), ptr<void>(cit), ptr<int32_t>(offsets_t),
                           ptr<int32_t>(bot), ptr<void>(ws), bytes, stream_of(ci)));
  return {cit, offsets_t, bot};
}

// offsets, row_indices, column_indices, offsets_t, column_indices_t, block_offsets_t and, with_plan, the fusion plan
std::tuple<Tensor, Tensor, Tensor, Tensor, Tensor, Tensor, OptTensor> dmoe_topology(const Tensor& padded_bins, int blocking, int64_t block_rows,
                                                                                    int64_t width, bool int32_indices, bool with_plan) {
  need_gpu(padded_bins);
  require(padded_bins.dim() == 1 && padded_bins.numel() > 0, "padded_bins holds one number per expert");
  const c10::DeviceGuard guard(padded_bins.device());
  const Tensor bins = offsets32(padded_bins);
  const int64_t experts = bins.numel(), nnz = block_rows * width;
  const auto ints = bins.options(), idx = ints.dtype(int32_indices ? at::kInt : at::kShort);
  Tensor offsets = at::empty({block_rows + 1}, ints), offsets_t = at::empty({experts * width + 1}, ints), ri = at::empty({nnz}, idx),
         ci = at::empty({nnz}, idx), cit = at::empty({nnz}, idx), bot = at::empty({nnz}, ints);
  OptTensor plan;
  size_t bytes = 0;
  if (with_plan) {
    bytes = stk_plan_bytes(block_rows, experts * width, nnz);
    plan = at::empty({(int64_t)bytes}, ints.dtype(at::kByte));
  }
  check(stk_dmoe_topology_plan(ptr<int32_t>(bins), experts, blocking, block_rows, width, int32_indices ? STK_I32 : STK_I16, ptr<int32_t>(offsets), ptr<void>(ri),
                               ptr<void>(ci), ptr<int32_t>(offsets_t), ptr<void>(cit), ptr<int32_t>(bot), ptr<uint8_t>(plan), bytes, stream_of(bins)));
  return {offsets, ri, ci, offsets_t, cit, bot, plan};
}

int elem_bytes(const Tensor& t) {
  if (t.element_size() != 2 && t.element_size() != 4)
    raise(PyExc_NotImplementedError, std::string("stk_amd: format conversion handles 2- and 4-byte elements, got ") + c10::toString(t.scalar_type()));
  return (int)t.element_size();
}

Tensor to_dense(const Tensor& data_, const Tensor& row_indices, const Tensor& column_indices, int64_t rows, int64_t cols, const OptTensor& offsets) {
  need_gpu(data_);
  const c10::DeviceGuard guard(data_.device());
  const Tensor data = data_.detach().contiguous(), ri = index(row_indices), ci = index(column_indices);
  Tensor out = at::empty({rows, cols}, data.options());
  const int64_t blocking = data.size(-1);
  const bool by_rows = offsets && offsets->scalar_type() == at::kInt && offsets->is_contiguous() && offsets->device() == data.device() && blocking > 0 &&
                       ci.numel() == data.size(0) && rows % blocking == 0 && offsets->numel() == rows / blocking + 1;
  check(stk_to_dense_rows(ptr<void>(data), by_rows ? ptr<int32_t>(*offsets) : nullptr, ptr<void>(ri), ptr<void>(ci), data.size(0), (int)blocking, rows, cols,
                          elem_bytes(data), index_dtype(ci.scalar_type()), ptr<void>(out), stream_of(data)));
  return out;
}

// Scratch allocations of this size or more are not left alive behind the small views returned.
constexpr int64_t kKeepBytes = 1 << 16;

// data, row_indices, column_indices and offsets of the nonzero blocks of x, and for matrices of few blocks, where they come
// with the rest, column_indices_t, offsets_t and block_offsets_t
std::tuple<Tensor, Tensor, Tensor, Tensor, OptTensor, OptTensor, OptTensor> to_sparse(const Tensor& x_, int64_t blocking, bool int32_indices) {
  need_gpu(x_);
  require(x_.dim() == 2, "to_sparse takes a matrix");
  const int64_t rows = x_.size(0), cols = x_.size(1);
  require(blocking > 0 && rows % blocking == 0 && cols % blocking == 0, "the matrix must be made of whole blocks");
  const c10::DeviceGuard guard(x_.device());
  const Tensor x = (x_.stride(1) != 1 && cols > 1 ? x_.contiguous() : x_).detach();
  const int64_t br = rows / blocking, bc = cols / blocking, blocks = br * bc;
  const hipStream_t stream = stream_of(x);
  if (capture_id(reinterpret_cast<int64_t>(stream)))
    raise(PyExc_RuntimeError, "to_sparse sizes its result by the number of nonzero blocks, which the host reads back: it cannot be captured into a graph");
  const int bytes = elem_bytes(x), idx = int32_indices ? STK_I32 : STK_I16;
  const bool small = blocks > 0 && blocks <= STK_TO_SPARSE_INDEX_BLOCKS && br <= 1024 && bc <= 1024;
  // one allocation for offsets (int32) and the block mask (bytes) behind it
  Tensor scratch = at::empty({4 * (br + 1) + std::max<int64_t>(blocks, 1)}, x.options().dtype(at::kByte));
  Tensor offsets = scratch.narrow(0, 0, 4 * (br + 1)).view(at::kInt);
  uint8_t* mask = ptr<uint8_t>(scratch) + 4 * (br + 1);
  // the index arrays need no nnz: launched before the host knows it, into room for every block (the first nnz entries are
  // written; the index tensors returned are views of that room, at multiples of 256 bytes like allocations of their own)
  const int64_t half = std::max<int64_t>((blocks + 127) / 128 * 128, 128), columns = (bc + 1 + 63) / 64 * 64;
  Tensor room = at::empty({(small ? 3 : 2) * half}, x.options().dtype(int32_indices ? at::kInt : at::kShort)), room_t;
  const auto third = [&](int i) { return ptr<char>(room) + i * half * room.element_size(); };
  const Mailbox box(x.device());
  int coordinates = STK_OK;
  if (small) {
    room_t = at::empty({columns + half}, x.options().dtype(at::kInt));
    check(stk_to_sparse_index(ptr<void>(x), rows, cols, x.stride(0), (int)blocking, bytes, mask, ptr<int32_t>(offsets), third(0), third(1),
                              ptr<int32_t>(room_t), third(2), ptr<int32_t>(room_t) + columns, idx, const_cast<int32_t*>(box.word), stream));
  } else {
    check(stk_to_sparse_count_nnz(ptr<void>(x), rows, cols, x.stride(0), (int)blocking, bytes, mask, ptr<int32_t>(offsets), const_cast<int32_t*>(box.word), stream));
    coordinates = stk_to_sparse_coordinates(rows, cols, (int)blocking, mask, ptr<int32_t>(offsets), third(0), third(1), idx, stream);
  }
  const int64_t nnz = box.receive(stream);   // (also where a launch behind the count's failed: the word is free only once it is delivered)
  check(coordinates);
  Tensor data = at::empty({nnz, blocking, blocking}, x.options());
  check(stk_to_sparse_gather(ptr<void>(x), rows, cols, x.stride(0), (int)blocking, bytes, third(0), third(1), nnz, idx, ptr<void>(data), stream));
  Tensor ri = room.narrow(0, 0, nnz), ci = room.narrow(0, half, nnz);
  OptTensor ci_t, offsets_t, bo_t;
  if (small) ci_t = room.narrow(0, 2 * half, nnz), offsets_t = room_t.narrow(0, 0, bc + 1), bo_t = room_t.narrow(0, columns, nnz);
  // A Matrix keeps these tensors for as long as it lives.  Where the room for every block is much more than the
  // nonzero blocks need (a large, very sparse matrix), they are copied out of it, and the offsets out of the
  // allocation they share with the block mask, so that the O(rows x columns / blocking^2) buffers can go.
  if (room.numel() * room.element_size() >= kKeepBytes && 4 * nnz <= blocks) {
    ri = ri.clone(), ci = ci.clone();
    if (small) ci_t = ci_t->clone(), offsets_t = offsets_t->clone(), bo_t = bo_t->clone();
  }
  if (scratch.numel() >= kKeepBytes && 16 * (br + 1) <= scratch.numel()) offsets = offsets.clone();
  return {data, ri, ci, offsets, ci_t, offsets_t, bo_t};
}

// ------------------------------------------------------------------------------------------------ values and routing
Tensor activation_product(const Tensor& sums_, const OptTensor& factor_, int activation) {
  need_gpu(sums_);
  const c10::DeviceGuard guard(sums_.device());
  const Tensor sums = sums_.detach().contiguous();
  Tensor out = at::empty_like(sums);
  OptTensor factor;
  if (factor_) {
    need_gpu(*factor_);
    factor = factor_->detach().contiguous();
    require(factor->sizes() == sums.sizes() && factor->scalar_type() == sums.scalar_type(), "sums and factor must have one shape and dtype");
  }
  if (sums.numel() == 0) return out;
  check(stk_activation_product(ptr<void>(sums), ptr<void>(factor), ptr<void>(out), sums.numel(), activation, value_dtype(sums), stream_of(sums)));
  return out;
}

// indices, bin_ids, bins, padded_bins, slot_rows, row_slots.  padded_rows < 0: row_slots gets exactly the rows of the
// padded layout, whose number the host waits for.
std::tuple<Tensor, Tensor, Tensor, Tensor, Tensor, Tensor> route(const Tensor& top_experts, int64_t experts, int64_t blocking, int64_t padded_rows) {
  need_gpu(top_experts);
  const c10::DeviceGuard guard(top_experts.device());
  const Tensor e = top_experts.reshape({-1}).to(at::kInt).contiguous();
  const int64_t slots = e.numel();
  const bool exact = padded_rows < 0;
  const int64_t rows = exact ? (slots + experts * (blocking - 1)) / std::max<int64_t>(blocking, 1) * blocking : padded_rows;
  const int64_t ws = ((int64_t)stk_route_workspace_bytes(slots, experts) + 3) / 4;
  // one allocation for the six outputs and the workspace
  Tensor all = at::empty({3 * slots + 2 * experts + rows + ws}, e.options());
  int64_t used = 0;
  const auto part = [&](int64_t n) {
    Tensor t = all.narrow(0, used, n);
    used += n;
    return t;
  };
  Tensor indices = part(slots), bin_ids = part(slots), slot_rows = part(slots), bins = part(experts), padded_bins = part(experts), row_slots = part(rows);
  const hipStream_t stream = stream_of(e);
  if (exact && capture_id(reinterpret_cast<int64_t>(stream)))
    raise(PyExc_RuntimeError, "route sizes the padded layout by the expert choices, which the host reads back: under a graph capture give it padded_rows");
  std::optional<Mailbox> box;
  if (exact) box.emplace(e.device());
  check(stk_route_total(ptr<int32_t>(e), slots, experts, (int)blocking, rows, ptr<int32_t>(indices), ptr<int32_t>(bin_ids), ptr<int32_t>(bins),
                        ptr<int32_t>(padded_bins), ptr<int32_t>(slot_rows), ptr<int32_t>(row_slots), ptr<int32_t>(all) + used, (size_t)ws * 4,
                        box ? const_cast<int32_t*>(box->word) : nullptr, stream));
  if (exact) row_slots = row_slots.narrow(0, 0, box->receive(stream));
  return {indices, bin_ids, bins, padded_bins, slot_rows, row_slots};
}

// 2-D 16-bit tensor whose rows the copy kernels can read in place (unit column stride, rows at multiples of 16 bytes);
// anything else is copied to row-major first.
Tensor rows16(const Tensor& x_) {
  const Tensor x = x_.detach();
  require(x.dim() == 2, "token rows are a matrix");
  if (x.numel() && !(x.stride(1) == 1 && x.stride(0) % 8 == 0 && x.stride(0) >= x.size(1) && aligned(x))) return x.contiguous();
  return x;
}
int64_t row_stride(const Tensor& x) { return x.numel() && x.size(0) > 1 ? x.stride(0) : std::max<int64_t>(x.size(1), 1); }
OptTensor weights32(const OptTensor& weights, int64_t slots) {
  if (!weights) return {};
  if (weights->numel() > 0) need_gpu(*weights);   // (a kernel reads them: an address in host memory would be a fault)
  Tensor w = weights->detach().reshape({-1}).to(at::kFloat).contiguous();
  if (w.numel() != slots)
    raise(PyExc_AssertionError, "one weight per slot: " + std::to_string(w.numel()) + " weights for " + std::to_string(slots) + " slots");
  return w;
}

// out[r] = (weights[s]) * x[s / top_k], s = row_slots[r]; zeros where s < 0
Tensor padded_gather(const Tensor& x_, const Tensor& row_slots, int top_k, const OptTensor& weights) {
  need_gpu(x_), need_gpu(row_slots);
  const c10::DeviceGuard guard(x_.device());
  const Tensor x = rows16(x_);
  const int64_t tokens = x.size(0), cols = x.size(1), rows = row_slots.numel();
  const OptTensor w = weights32(weights, tokens * top_k);
  Tensor out = at::empty({rows, cols}, x.options());
  check(stk_padded_gather(ptr<void>(x), tokens, cols, row_stride(x), ptr<int32_t>(row_slots), ptr<float>(w), top_k, rows, ptr<void>(out),
                          std::max<int64_t>(cols, 1), value_dtype(x), stream_of(x)));
  return out;
}

// out[t] = sum_k (weights[s]) * x[slot_rows[s]], s = t * top_k + k
Tensor padded_scatter(const Tensor& x_, const Tensor& slot_rows, int top_k, const OptTensor& weights) {
  need_gpu(x_), need_gpu(slot_rows);
  const c10::DeviceGuard guard(x_.device());
  const Tensor x = rows16(x_);
  const int64_t rows = x.size(0), cols = x.size(1), slots = slot_rows.numel();
  if (top_k < 1 || slots % top_k)
    raise(PyExc_AssertionError, std::to_string(slots) + " slots are not a multiple of top_k = " + std::to_string(top_k));
  const OptTensor w = weights32(weights, slots);
  Tensor out = at::empty({slots / top_k, cols}, x.options());
  check(stk_padded_scatter(ptr<void>(x), rows, cols, row_stride(x), ptr<int32_t>(slot_rows), ptr<float>(w), top_k, slots / top_k, ptr<void>(out),
                           std::max<int64_t>(cols, 1), value_dtype(x), stream_of(x)));
  return out;
}

// fp32 [slots]: <x[slot_rows[s]], grad[s / top_k]>
Tensor padded_scatter_weight_gradient(const Tensor& x_, const Tensor& grad_, const Tensor& slot_rows, int top_k) {
  need_gpu(x_), need_gpu(grad_), need_gpu(slot_rows);
  const c10::DeviceGuard guard(x_.device());
  const Tensor x = rows16(x_), grad = rows16(grad_);
  require(x.scalar_type() == grad.scalar_type() && x.size(1) == grad.size(1), "x and grad must have one dtype and row length");
  const int64_t slots = slot_rows.numel();
  require(grad.size(0) * top_k == slots, "one gradient row per token");
  Tensor out = at::empty({slots}, x.options().dtype(at::kFloat));
  check(stk_padded_scatter_weight_gradient(ptr<void>(x), x.size(0), x.size(1), row_stride(x), ptr<void>(grad), row_stride(grad), ptr<int32_t>(slot_rows),
                                           top_k, grad.size(0), ptr<float>(out), value_dtype(x), stream_of(x)));
  return out;
}

// out = act(sdd(padded_gather(x), rhs)); false, with nothing launched, when the library has no such kernel for this case
bool sdd_gather(const Tensor& x_, const Tensor& row_slots, int top_k, const Tensor& rhs_, int64_t m, int64_t n, const Tensor& out, const Tensor& offsets,
                const Tensor& row_indices, const Tensor& column_indices, const OptTensor& plan, int activation) {
  need_gpu(x_), need_gpu(row_slots), need_gpu(rhs_), need_gpu(out);
  const int64_t b = out.size(-1), nnz = row_indices.numel();
  const c10::DeviceGuard guard(out.device());
  const Tensor x = rows16(x_);
  const int64_t tokens = x.size(0), k = x.size(1);
  require(rhs_.dim() == 2 && k == rhs_.size(0) && n == rhs_.size(1), "incompatible dimensions");
  require(row_slots.scalar_type() == at::kInt && row_slots.is_contiguous() && row_slots.numel() >= m, "row_slots must name the rows of the padded layout");
  matmul_dims(m, k, n, b);
  if (tokens == 0 || tokens * row_stride(x) * 2 >= (int64_t(1) << 32)) return false;
  if (nnz == 0) return true;
  const Tensor rhs = dense_operand(rhs_);
  require(out.is_contiguous() && x.scalar_type() == rhs.scalar_type() && x.scalar_type() == out.scalar_type(), "operands and out must have one dtype");
  const Tensor ri = index(row_indices), ci = index(column_indices), offs = offsets32(offsets);
  const int status = stk_sdd_gather(ptr<void>(x), tokens, row_stride(x), ptr<int32_t>(row_slots), top_k, ptr<void>(rhs), rhs.stride(0), rhs.stride(1), m, k, n,
                                    ptr<void>(out), plan ? ptr<int32_t>(offs) : nullptr, ptr<void>(ri), ptr<void>(ci), nnz, (int)b, value_dtype(out),
                                    index_dtype(ri.scalar_type()), ptr<uint8_t>(plan), activation, stream_of(out));
  if (status == STK_ERR_UNSUPPORTED) return false;
  check(status);
  return true;
}

// out = padded_scatter(sparse @ rhs, top_k = 1, weights); the status, STK_ERR_UNSUPPORTED, with nothing launched, when the
// library has no such kernel
int dsd_scatter(int64_t m, int64_t k, const Tensor& data, const Tensor& offsets, const Tensor& column_indices, const Tensor& rhs_, const Tensor& row_slots,
                 const OptTensor& weights, const Tensor& out, const Tensor& plan, const OptTensor& workspace) {
  need_gpu(data), need_gpu(rhs_), need_gpu(row_slots), need_gpu(out);
  require(rhs_.dim() == 2 && k == rhs_.size(0), "incompatible dimensions");
  const int64_t n = rhs_.size(1), b = data.size(-1);
  matmul_dims(m, k, n, b);
  const c10::DeviceGuard guard(out.device());
  const Tensor rhs = dense_operand(rhs_);
  require(data.is_contiguous() && out.stride(1) == 1 && out.size(1) == n, "the sparse values must be contiguous and out row-major");
  require(data.scalar_type() == rhs.scalar_type() && data.scalar_type() == out.scalar_type(), "operands and out must have one dtype");
  require(row_slots.scalar_type() == at::kInt && row_slots.is_contiguous() && row_slots.numel() >= m, "row_slots must name the rows of the padded layout");
  const OptTensor w = weights32(weights, out.size(0));
  const Tensor ci = index(column_indices), offs = offsets32(offsets);
  return stk_dsd_scatter(m, k, n, ptr<void>(data), ptr<int32_t>(offs), ptr<void>(ci), ptr<void>(rhs), rhs.stride(0), rhs.stride(1),
                         ptr<int32_t>(row_slots), ptr<float>(w), out.size(0), ptr<void>(out), out.stride(0), data.size(0), (int)b, value_dtype(out),
                         index_dtype(ci.scalar_type()), ptr<uint8_t>(plan), ptr<void>(workspace), workspace ? workspace->numel() : 0,
                         stream_of(out));
}

// Whether dsd_scatter_few is for these sizes (-1: no), and the size of the workspace, with room for `partial_tiles`, of the
// stk_dsd whose bits it gives, 0 if that one cuts no tile.
int64_t dsd_scatter_few_case(int64_t m, int64_t n, int64_t nnz, int64_t slots, int64_t partial_tiles) {
  if (stk_dsd_scatter_few_bytes(m, n, nnz, slots) == 0) return -1;
  const int64_t bytes = partial_tiles > 0 ? stk_dsd_workspace_counter_bytes() + partial_tiles * stk_dsd_workspace_slot_bytes() : 0;
  return stk_dsd_cuts(m, n, nnz, bytes) ? bytes : 0;
}

// padded_scatter(sparse @ rhs, top_k, weights) where the block rows hold few slots each; nothing, with nothing launched, when the
// library has no kernel for this case
OptTensor dsd_scatter_few(int64_t m, int64_t k, const Tensor& data, const Tensor& offsets, const Tensor& column_indices, const Tensor& rhs_,
                          const Tensor& row_slots, const Tensor& slot_rows, int top_k, const OptTensor& weights, const OptTensor& plan,
                          int64_t dsd_workspace_bytes) {
  // (what the two calls refuse is left to them)
  if (rhs_.dim() != 2 || k != rhs_.size(0) || top_k < 1) return {};
  const int64_t n = rhs_.size(1), b = data.size(-1), slots = slot_rows.numel(), nnz = data.size(0);
  for (const Tensor* t : {&rhs_, &row_slots, &slot_rows, &offsets, &column_indices})
    if (t->device() != data.device()) return {};
  for (const Tensor* t : {&row_slots, &slot_rows})
    if (t->scalar_type() != at::kInt || !t->is_contiguous()) return {};
  if (b != 128 || n % b || slots % top_k || data.scalar_type() != rhs_.scalar_type() || !data.is_contiguous() || !aligned(data) || row_slots.numel() < m ||
      (data.scalar_type() != at::kHalf && data.scalar_type() != at::kBFloat16))
    return {};
  const int64_t bytes = stk_dsd_scatter_few_bytes(m, n, nnz, slots);
  if (bytes == 0) return {};
  const c10::DeviceGuard guard(rhs_.device());
  const Tensor rhs = dense_operand(rhs_);
  const OptTensor w = weights32(weights, slots);
  const Tensor ci = index(column_indices), offs = offsets32(offsets);
  Tensor out = at::empty({slots / top_k, n}, rhs.options());
  const Tensor sums = at::empty({bytes / 4}, rhs.options().dtype(at::kFloat));
  const int status = stk_dsd_scatter_few_as_cut(m, k, n, ptr<void>(data), ptr<int32_t>(offs), ptr<void>(ci), ptr<void>(rhs), rhs.stride(0), rhs.stride(1),
                                         ptr<int32_t>(row_slots), ptr<int32_t>(slot_rows), ptr<float>(w), top_k, slots / top_k, ptr<void>(out), n, nnz,
                                         (int)b, value_dtype(rhs), index_dtype(ci.scalar_type()), ptr<void>(sums), bytes,
                                                ptr<uint8_t>(plan), dsd_workspace_bytes, stream_of(rhs));
  if (status == STK_ERR_UNSUPPORTED) return {};
  check(status);
  return out;
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.def("abi_version", [] { return STK_AMD_ABI_VERSION; });
  m.def("sdd", &sdd, py::call_guard<py::gil_scoped_release>());
  m.def("dsd", &dsd, py::call_guard<py::gil_scoped_release>());
  m.def("dds", &dds, py::call_guard<py::gil_scoped_release>());
  m.def("dsd_dds", &dsd_dds, py::call_guard<py::gil_scoped_release>());
  m.def("dsd_dsd", &dsd_dsd, py::call_guard<py::gil_scoped_release>());
  m.def("sdd_dsd", &sdd_dsd, py::call_guard<py::gil_scoped_release>());
  m.def("build_plan", &build_plan, py::call_guard<py::gil_scoped_release>());
  m.def("capture_id", &capture_id, py::call_guard<py::gil_scoped_release>());
  m.def("follow", &follow, py::call_guard<py::gil_scoped_release>());
  m.def("row_indices", &row_indices, py::call_guard<py::gil_scoped_release>());
  m.def("transpose_meta", &transpose_meta, py::call_guard<py::gil_scoped_release>());
  m.def("dmoe_topology", &dmoe_topology, py::call_guard<py::gil_scoped_release>());
  m.def("to_dense", &to_dense, py::call_guard<py::gil_scoped_release>());
  m.def("to_sparse", &to_sparse, py::call_guard<py::gil_scoped_release>());
  m.def("activation_product", &activation_product, py::call_guard<py::gil_scoped_release>());
  m.def("route", &route, py::call_guard<py::gil_scoped_release>());
  m.def("padded_gather", &padded_gather, py::call_guard<py::gil_scoped_release>());
  m.def("padded_scatter", &padded_scatter, py::call_guard<py::gil_scoped_release>());
  m.def("padded_scatter_weight_gradient", &padded_scatter_weight_gradient, py::call_guard<py::gil_scoped_release>());
  m.def("sdd_gather", &sdd_gather, py::call_guard<py::gil_scoped_release>());
  m.def("sdd_gather_reads_plan", &stk_sdd_gather_reads_plan);
  m.def("dsd_scatter_few_case", &dsd_scatter_few_case);
  m.def("dsd_scatter_few", &dsd_scatter_few, py::call_guard<py::gil_scoped_release>());
  m.def("dsd_scatter", &dsd_scatter, py::call_guard<py::gil_scoped_release>());
}
