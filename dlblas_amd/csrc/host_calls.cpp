// The host side of the Python entry points as one native call each: argument checks, output allocation, workspace lookup
// and the C ABI call.  A decode-sized GEMM runs 5 us on the GPU; through the Python wrapper, torch.library.custom_op and
// ctypes its launch took 20 us of host time, a quantise + GEMM pair 45 us, an expert MLP of four kernels 186 us, so the GPU
// waited for the host (1 x 2112 x 7168: 19.6 us per call, 6.0 us of it the kernel).
//
// Every function takes the arguments of the Python function of its name and either does the call or returns None without
// having enqueued anything.  None means "not a plain call": tensor subclasses, dispatch and function modes, tracing, inputs
// that require grad or carry a tangent, arguments the checks refuse, layouts only the Python path handles.  The Python function then goes on as
// it would without this module, through its custom op and its own checks and messages.
#include <Python.h>

#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/core/Tensor.h>
#include <ATen/hip/EmptyTensor.h>
#include <ATen/record_function.h>
#include <c10/core/DefaultDtype.h>
#include <c10/core/GradMode.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/autograd/python_variable.h>

#include <algorithm>
#include <cstdint>
#include <cstring>
#include <string>
#include <unordered_map>
#include <utility>
#include <vector>

#include "../../include/dlblas_fp8_gemm.h"
#include "../../include/dlblas_fp8_moe.h"

namespace {

constexpr int64_t kBlock = 128;

// The entry points of the library that ctypes has loaded, by address (init() below): one library, whichever was chosen.
struct Abi {
  decltype(&dlb_last_error) last_error;
  decltype(&dlb_workspace_lock) lock;
  decltype(&dlb_workspace_unlock) unlock;
  decltype(&dlb_fp8_gemm) gemm;
  decltype(&dlb_fp8_gemm_grouped_contiguous) contiguous;
  decltype(&dlb_fp8_gemm_grouped_contiguous_same_rows) contiguous_same_rows;
  decltype(&dlb_fp8_gemm_grouped_contiguous_gather_silu_quant) contiguous_gather_act;
  decltype(&dlb_fp8_gemm_grouped_masked) masked;
  decltype(&dlb_expert_gate_up_masked) masked_act;
  decltype(&dlb_fp8_gemm_grouped_ragged) ragged;
  decltype(&dlb_expert_gate_up_ragged) ragged_act;
  decltype(&dlb_expert_plan) plan;
  decltype(&dlb_fp8_quant_group) quant_group;
  decltype(&dlb_silu_mul_quant_masked) silu_masked;
  decltype(&dlb_ep_scatter_workspace_bytes) scatter_ws;
  decltype(&dlb_ep_scatter_rows_host) scatter_rows;
  decltype(&dlb_ep_gather) gather;
} abi;
PyObject* g_make_workspace = nullptr;  // _lib.workspace: creates and keeps the buffer of a (device, stream)

// ---- what a plain call is ---------------------------------------------------------------------------------------------

const c10::DispatchKeySet kPlainKeys({c10::DispatchKey::CUDA, c10::DispatchKey::AutogradCUDA, c10::DispatchKey::ADInplaceOrView, c10::DispatchKey::AutocastCUDA});
const c10::DispatchKeySet kPlainIncluded({c10::DispatchKey::BackendSelect, c10::DispatchKey::ADInplaceOrView, c10::DispatchKey::AutocastCUDA});

// (raw bits: set difference on DispatchKeySet leaves the backend bits alone)
bool within(c10::DispatchKeySet keys, c10::DispatchKeySet allowed) { return (keys.raw_repr() & ~allowed.raw_repr()) == 0; }

bool no_modes() { return within(c10::impl::tls_local_dispatch_key_set().included_, kPlainIncluded) && !at::impl::torch_function_mode_enabled(); }

// A dense GPU tensor that nothing but its own storage stands behind; nullptr otherwise.
const at::Tensor* plain(PyObject* o) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  if (!t.defined() || !t.is_cuda() || !within(t.key_set(), kPlainKeys)) return nullptr;
  if (t.is_conj() || t.is_neg() || (c10::GradMode::is_enabled() && t.requires_grad()) || t._fw_grad(0).defined()) return nullptr;
  return &t;
}

template <size_t N>
bool all_plain(PyObject* const* args, const at::Tensor* (&out)[N]) {
  if (!no_modes()) return false;
  for (size_t i = 0; i < N; ++i) {
    out[i] = plain(args[i]);
    if (!out[i] || out[i]->get_device() != out[0]->get_device()) return false;
  }
  return true;
}

// Makes the tensors' device current for the scope (a no-op in the usual case).
struct DeviceScope {
  c10::DeviceIndex before, dev;
  explicit DeviceScope(const at::Tensor& t) : before(c10::hip::current_device()), dev(t.get_device()) {
    if (dev != before) c10::hip::set_device(dev);
  }
  ~DeviceScope() {
    if (dev != before) c10::hip::set_device(before);
  }
};

struct Workspace {
  void* ptr;
  size_t bytes;
};

// The buffer of (device, stream), the same one the ctypes path uses: _lib.workspace() makes it, this map remembers it.  The
// map holds a reference, so an entry stays valid; it is guarded by the GIL, which every caller holds.
bool workspace_of(c10::DeviceIndex dev, hipStream_t stream, const at::Tensor& like, Workspace* ws) {
  struct Hash {
    size_t operator()(const std::pair<int, void*>& k) const { return std::hash<void*>()(k.second) * 31 + k.first; }
  };
  static auto* cache = new std::unordered_map<std::pair<int, void*>, at::Tensor, Hash>();
  const std::pair<int, void*> key(dev, stream);
  auto found = cache->find(key);
  if (found == cache->end()) {
    PyObject* wrapped = THPVariable_Wrap(like);
    PyObject* device = wrapped ? PyObject_GetAttrString(wrapped, "device") : nullptr;
    Py_XDECREF(wrapped);
    if (!device) return false;
    PyObject* buf = PyObject_CallFunction(g_make_workspace, "OK", device, static_cast<unsigned long long>(reinterpret_cast<uintptr_t>(stream)));
    Py_DECREF(device);
    if (!buf) return false;
    found = cache->emplace(key, THPVariable_Unpack(buf)).first;
    Py_DECREF(buf);
  }
  ws->ptr = found->second.data_ptr();
  ws->bytes = static_cast<size_t>(found->second.numel());
  return true;
}

hipStream_t stream_of(const at::Tensor& t) { return c10::hip::getCurrentHIPStream(t.get_device()).stream(); }

at::Tensor empty(at::IntArrayRef size, at::ScalarType dtype, const at::Tensor& like) {
  return at::Tensor(at::detail::empty_cuda(size, dtype, like.device(), std::nullopt));
}
at::Tensor empty_strided(at::IntArrayRef size, at::IntArrayRef stride, at::ScalarType dtype, const at::Tensor& like) {
  return at::Tensor(at::detail::empty_strided_cuda(size, stride, dtype, like.device()));
}

// A custom op that mutates an argument moves its version counter on.
void written(const at::Tensor& t) {
  if (!t.is_inference()) t.unsafeGetTensorImpl()->bump_version();
}

void* ptr(const at::Tensor& t) { return t.numel() > 0 ? t.data_ptr() : nullptr; }
float* fptr(const at::Tensor& t) { return static_cast<float*>(ptr(t)); }
int32_t* iptr(const at::Tensor& t) { return static_cast<int32_t*>(ptr(t)); }
int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

bool is_f8(const at::Tensor& t) { return t.scalar_type() == at::kFloat8_e4m3fn; }
bool is_f32(const at::Tensor& t) { return t.scalar_type() == at::kFloat; }
int out_code(at::ScalarType t) { return t == at::kBFloat16 ? DLB_OUT_BF16 : t == at::kFloat ? DLB_OUT_F32 : -1; }
int in_code(at::ScalarType t) { return t == at::kBFloat16 ? DLB_IN_BF16 : t == at::kHalf ? DLB_IN_F16 : t == at::kFloat ? DLB_IN_F32 : -1; }
int idx_code(at::ScalarType t) { return t == at::kInt ? DLB_IDX_I32 : t == at::kLong ? DLB_IDX_I64 : -1; }

// An op event of torch's profiler, as the custom ops of the Python path leave one; nothing when nobody records.
struct OpRecord {
  at::RecordFunction guard{at::RecordScope::FUNCTION};
  std::vector<c10::IValue> inputs;
  template <size_t N>
  OpRecord(const char* name, const at::Tensor* const (&t)[N]) {
    if (!guard.isActive()) return;
    if (guard.needsInputs())
      for (const at::Tensor* x : t) inputs.emplace_back(*x);
    guard.before(name, c10::ArrayRef<const c10::IValue>(inputs.data(), inputs.size()));
  }
};

// Allocations and launches run without the GIL: a launch waits while the hardware queue is full.  No Python object is touched
// in such a scope.
class NoGil {
 public:
  NoGil() : state_(PyEval_SaveThread()) {}
  ~NoGil() { PyEval_RestoreThread(state_); }
  NoGil(const NoGil&) = delete;
  NoGil& operator=(const NoGil&) = delete;

 private:
  PyThreadState* state_;
};

// Keeps the launches of several library calls on one workspace together.  Inside a NoGil scope only: a thread that waits for
// the lock must not keep its holder from finishing.
class Together {
 public:
  explicit Together(const Workspace& ws) : ws_(ws.ptr) { abi.lock(ws_); }
  ~Together() { abi.unlock(ws_); }
  Together(const Together&) = delete;
  Together& operator=(const Together&) = delete;

 private:
  const void* ws_;
};

// After the first launch of a chain there is no way back to the Python path.
PyObject* launch_failed(int rc) {
  return PyErr_Format(PyExc_RuntimeError, "dlblas fp8_gemm error %d: %s", rc, abi.last_error());
}

#define NOT_PLAIN Py_RETURN_NONE
#define HANDLE_EXCEPTIONS_BEGIN try {
#define HANDLE_EXCEPTIONS_END                          \
  }                                                    \
  catch (const c10::OutOfMemoryError& e) {             \
    NOT_PLAIN; /* the Python path raises torch's own */ \
  }                                                    \
  catch (const std::exception& e) {                    \
    PyErr_SetString(PyExc_RuntimeError, e.what());     \
    return nullptr;                                    \
  }

// ---- dense ------------------------------------------------------------------------------------------------------------

// fp8_gemm(a, b, a_s, b_s) -> c
PyObject* fp8_gemm(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_EXCEPTIONS_BEGIN
  const at::Tensor* t[4];
  if (n != 4 || !all_plain(args, t)) NOT_PLAIN;
  const at::Tensor &a = *t[0], &b = *t[1], &a_s = *t[2], &b_s = *t[3];
  const at::ScalarType out = c10::get_default_dtype_as_scalartype();
  if (out_code(out) < 0 || !is_f8(a) || !is_f8(b) || !is_f32(a_s) || !is_f32(b_s) || b.dim() != 2 || a.dim() < 1 || b_s.dim() != 2 || a_s.dim() < 1)
    NOT_PLAIN;
  if (!a.is_contiguous() || !b.is_contiguous() || !a_s.is_contiguous() || !b_s.is_contiguous()) NOT_PLAIN;
  const int64_t K = b.size(1), N = b.size(0), kb = ceil_div(K, kBlock);
  if (K == 0 || N == 0 || a.size(-1) != K) NOT_PLAIN;
  const int64_t M = a.numel() / K;
  if (M == 0 || a_s.numel() != M * kb || a_s.size(-1) != kb || b_s.size(0) != ceil_div(N, kBlock) || b_s.size(1) != kb) NOT_PLAIN;
  const OpRecord record("dlblas::fp8_gemm", t);
  DeviceScope scope(a);
  const hipStream_t stream = stream_of(a);
  Workspace ws;
  if (!workspace_of(scope.dev, stream, a, &ws)) return nullptr;
  at::DimVector size(a.sizes());
  size.back() = N;
  at::Tensor c;
  int rc;
  {
    const NoGil nogil;
    c = empty(size, out, a);
    rc = abi.gemm(ptr(a), ptr(b), fptr(a_s), fptr(b_s), ptr(c), M, N, K, kb, 1, out_code(out), ws.ptr, ws.bytes, stream);
  }
  if (rc != DLB_OK) NOT_PLAIN;
  return THPVariable_Wrap(std::move(c));
  HANDLE_EXCEPTIONS_END
}

// per_token_group_quant_fp8(x, group_size, eps, column_major_scales) -> (q, s)
PyObject* quant(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_EXCEPTIONS_BEGIN
  const at::Tensor* t[1];
  if (n != 4 || !all_plain(args, t)) NOT_PLAIN;
  const at::Tensor& x = *t[0];
  if (!PyLong_CheckExact(args[1]) || !PyFloat_CheckExact(args[2]) || !PyBool_Check(args[3])) NOT_PLAIN;
  const int64_t group = PyLong_AsLongLong(args[1]);
  if (PyErr_Occurred()) {
    PyErr_Clear();
    NOT_PLAIN;
  }
  const float eps = static_cast<float>(PyFloat_AS_DOUBLE(args[2]));
  const bool col_major = args[3] == Py_True;
  if (in_code(x.scalar_type()) < 0 || x.dim() < 2 || group <= 0 || x.stride(-1) != 1 || x.numel() == 0) NOT_PLAIN;
  const int64_t K = x.size(-1), rows = x.numel() / K;
  if (K % group != 0 || (x.dim() > 2 && !x.is_contiguous())) NOT_PLAIN;
  const OpRecord record("dlblas::per_token_group_quant_fp8", t);
  const int64_t groups = K / group;
  const int64_t row_stride = x.dim() == 2 ? x.stride(0) : K;
  DeviceScope scope(x);
  at::Tensor q, s;
  at::DimVector size(x.sizes());
  size.back() = groups;
  int rc;
  {
    const NoGil nogil;
    q = empty(x.sizes(), at::kFloat8_e4m3fn, x);
    if (col_major) {
      // a [groups, rows...] buffer viewed with the group axis last
      at::DimVector stride(x.dim(), 1);
      for (int64_t d = x.dim() - 3; d >= 0; --d) stride[d] = stride[d + 1] * size[d + 1];
      stride.back() = rows;
      s = empty_strided(size, stride, at::kFloat, x);
    } else {
      s = empty(size, at::kFloat, x);
    }
    rc = abi.quant_group(ptr(x), in_code(x.scalar_type()), ptr(q), fptr(s), rows, K, group, row_stride, col_major ? 1 : groups, col_major ? rows : 1,
                         eps, stream_of(x));
  }
  if (rc != DLB_OK) NOT_PLAIN;
  PyObject* out = PyTuple_New(2);
  if (!out) return nullptr;
  PyTuple_SET_ITEM(out, 0, THPVariable_Wrap(std::move(q)));
  PyTuple_SET_ITEM(out, 1, THPVariable_Wrap(std::move(s)));
  return out;
  HANDLE_EXCEPTIONS_END
}

// ---- grouped ----------------------------------------------------------------------------------------------------------

bool weights_ok(const at::Tensor& w, const at::Tensor& w_s) {
  return is_f8(w) && is_f32(w_s) && w.dim() == 3 && w_s.dim() == 3 && w.is_contiguous() && w_s.is_contiguous() && w.numel() > 0 &&
         w.size(2) % 16 == 0 && w_s.size(0) == w.size(0) && w_s.size(1) == ceil_div(w.size(1), kBlock) && w_s.size(2) == ceil_div(w.size(2), kBlock);
}

bool index_vector(const at::Tensor& t, int64_t n) { return t.scalar_type() == at::kInt && t.dim() == 1 && t.size(0) == n && t.is_contiguous(); }

// grouped_contiguous(a, a_s, w, w_s, out, m_indices) -> True
PyObject* grouped_contiguous(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_EXCEPTIONS_BEGIN
  const at::Tensor* t[6];
  if (n != 6 || !all_plain(args, t)) NOT_PLAIN;
  const at::Tensor &a = *t[0], &a_s = *t[1], &w = *t[2], &w_s = *t[3], &out = *t[4], &idx = *t[5];
  if (!weights_ok(w, w_s)) NOT_PLAIN;
  const int64_t G = w.size(0), N = w.size(1), K = w.size(2), kb = ceil_div(K, kBlock);
  if (!is_f8(a) || !is_f32(a_s) || out_code(out.scalar_type()) < 0 || a.dim() != 2 || a.size(1) != K || a_s.dim() != 2 || out.dim() != 2) NOT_PLAIN;
  const int64_t M = a.size(0);
  if (M == 0 || !a.is_contiguous() || !out.is_contiguous() || a_s.size(0) != M || a_s.size(1) != kb || out.size(0) != M || out.size(1) != N ||
      !index_vector(idx, M))
    NOT_PLAIN;
  const OpRecord record("dlblas::fp8_gemm_grouped_contiguous", t);
  DeviceScope scope(a);
  const hipStream_t stream = stream_of(a);
  Workspace ws;
  if (!workspace_of(scope.dev, stream, a, &ws)) return nullptr;
  int rc;
  {
    const NoGil nogil;
    rc = abi.contiguous(ptr(a), ptr(w), fptr(a_s), fptr(w_s), ptr(out), iptr(idx), M, N, K, static_cast<int32_t>(G), a_s.stride(0), a_s.stride(1),
                        out_code(out.scalar_type()), ws.ptr, ws.bytes, stream);
  }
  if (rc != DLB_OK) NOT_PLAIN;
  written(out);
  Py_RETURN_TRUE;
  HANDLE_EXCEPTIONS_END
}

bool masked_operand(const at::Tensor& a, const at::Tensor& a_s, int64_t G, int64_t K) {
  return is_f8(a) && is_f32(a_s) && a.dim() == 3 && a_s.dim() == 3 && a.size(0) == G && a.size(2) == K && a.is_contiguous() && a.numel() > 0 &&
         a_s.size(0) == G && a_s.size(1) == a.size(1) && a_s.size(2) == ceil_div(K, kBlock);
}

// grouped_masked(a, a_s, w, w_s, out, masked_m, expected_m) -> True
PyObject* grouped_masked(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_EXCEPTIONS_BEGIN
  const at::Tensor* t[6];
  if (n != 7 || !all_plain(args, t) || !PyLong_CheckExact(args[6])) NOT_PLAIN;
  const at::Tensor &a = *t[0], &a_s = *t[1], &w = *t[2], &w_s = *t[3], &out = *t[4], &mm = *t[5];
  if (!weights_ok(w, w_s)) NOT_PLAIN;
  const int64_t G = w.size(0), N = w.size(1), K = w.size(2);
  if (!masked_operand(a, a_s, G, K) || out_code(out.scalar_type()) < 0 || out.dim() != 3 || out.size(0) != G || out.size(1) != a.size(1) ||
      out.size(2) != N || !out.is_contiguous() || !index_vector(mm, G))
    NOT_PLAIN;
  const long hint = PyLong_AsLong(args[6]);
  if (PyErr_Occurred() || hint != static_cast<int32_t>(hint)) {
    PyErr_Clear();
    NOT_PLAIN;
  }
  const OpRecord record("dlblas::fp8_gemm_grouped_masked", t);
  DeviceScope scope(a);
  const hipStream_t stream = stream_of(a);
  Workspace ws;
  if (!workspace_of(scope.dev, stream, a, &ws)) return nullptr;
  int rc;
  {
    const NoGil nogil;
    rc = abi.masked(ptr(a), ptr(w), fptr(a_s), fptr(w_s), ptr(out), iptr(mm), static_cast<int32_t>(hint), a.size(1), N, K, static_cast<int32_t>(G),
                    a_s.stride(0), a_s.stride(1), a_s.stride(2), out_code(out.scalar_type()), ws.ptr, ws.bytes, stream);
  }
  if (rc != DLB_OK) NOT_PLAIN;
  written(out);
  Py_RETURN_TRUE;
  HANDLE_EXCEPTIONS_END
}

// ---- expert MLPs ------------------------------------------------------------------------------------------------------

// forms of dlb_expert_plan
enum Form : int { kStepsApart = 0, kOnRowRanges = 1, kOnWholeBlocks = 2 };

Form expert_form(int mode, int64_t rows, int64_t N, int64_t K, int64_t G, int64_t hint, bool quantising, const Workspace& ws) {
  int form = kStepsApart;
  if (abi.plan(mode, rows, N, K, static_cast<int32_t>(G), static_cast<int32_t>(hint), quantising, ws.bytes, 256, &form) != DLB_OK) return kStepsApart;
  return static_cast<Form>(form);
}

// low_latency_experts(a, a_s, w13, w13_s, w2, w2_s, masked_m, expected_m) -> down_output (bf16)
PyObject* low_latency_experts(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_EXCEPTIONS_BEGIN
  const at::Tensor* t[7];
  if (n != 8 || !all_plain(args, t) || !PyLong_CheckExact(args[7])) NOT_PLAIN;
  const at::Tensor &a = *t[0], &a_s = *t[1], &w13 = *t[2], &w13_s = *t[3], &w2 = *t[4], &w2_s = *t[5], &mm = *t[6];
  if (!weights_ok(w13, w13_s) || !weights_ok(w2, w2_s)) NOT_PLAIN;
  const int64_t G = w13.size(0), N = w13.size(1), K = w13.size(2), inter = N / 2, H = w2.size(1);
  if (!masked_operand(a, a_s, G, K) || N % (2 * kBlock) != 0 || K % kBlock != 0 || w2.size(0) != G || w2.size(2) != inter || !index_vector(mm, G)) NOT_PLAIN;
  const int64_t M = a.size(1);
  long hint = PyLong_AsLong(args[7]);
  if (PyErr_Occurred()) {
    PyErr_Clear();
    NOT_PLAIN;
  }
  hint = std::min<long>(hint, M);
  if (hint != static_cast<int32_t>(hint)) NOT_PLAIN;
  const OpRecord record("dlblas::low_latency_experts", t);
  DeviceScope scope(a);
  const hipStream_t stream = stream_of(a);
  Workspace ws;
  if (!workspace_of(scope.dev, stream, a, &ws)) return nullptr;
  const int32_t g = static_cast<int32_t>(G), m_hint = static_cast<int32_t>(hint);
  at::Tensor q, s, gate_up, out;
  int rc = DLB_OK;
  bool begun = false;  // something is enqueued: no way back to the Python path
  {
    const NoGil nogil;
    q = empty({G, M, inter}, at::kFloat8_e4m3fn, a);
    bool fused = false;
    if (expert_form(2, M, N, K, G, hint, true, ws) != kStepsApart) {
      // rows of a K block contiguous: what the second GEMM reads without a re-layout pass
      s = empty_strided({G, M, inter / kBlock}, {inter / kBlock * M, 1, M}, at::kFloat, a);
      fused = abi.masked_act(ptr(a), ptr(w13), fptr(a_s), fptr(w13_s), ptr(q), fptr(s), iptr(mm), m_hint, M, N, K, g, a_s.stride(0), a_s.stride(1),
                             a_s.stride(2), s.stride(0), s.stride(1), s.stride(2), 1e-10f, ws.ptr, ws.bytes, stream) == DLB_OK;
    }
    if (!fused) {
      gate_up = empty({G, M, N}, at::kBFloat16, a);
      rc = abi.masked(ptr(a), ptr(w13), fptr(a_s), fptr(w13_s), ptr(gate_up), iptr(mm), m_hint, M, N, K, g, a_s.stride(0), a_s.stride(1), a_s.stride(2),
                      DLB_OUT_BF16, ws.ptr, ws.bytes, stream);
      if (rc == DLB_OK) {
        begun = true;
        s = empty({G, M, inter / kBlock}, at::kFloat, a);
        rc = abi.silu_masked(ptr(gate_up), DLB_IN_BF16, ptr(q), fptr(s), iptr(mm), G, M, inter, s.stride(0), s.stride(1), s.stride(2), stream);
        gate_up.reset();
      }
    }
    if (rc == DLB_OK) {
      begun = true;
      out = empty({G, M, H}, at::kBFloat16, a);
      rc = abi.masked(ptr(q), ptr(w2), fptr(s), fptr(w2_s), ptr(out), iptr(mm), m_hint, M, H, inter, g, s.stride(0), s.stride(1), s.stride(2),
                      DLB_OUT_BF16, ws.ptr, ws.bytes, stream);
    }
  }
  if (rc != DLB_OK) {
    if (begun) return launch_failed(rc);
    NOT_PLAIN;
  }
  return THPVariable_Wrap(std::move(out));
  HANDLE_EXCEPTIONS_END
}

int gather(const at::Tensor& in, const at::Tensor& ids, const at::Tensor& weights, const at::Tensor& index, const at::Tensor& out, hipStream_t stream) {
  return abi.gather(ptr(in), in_code(in.scalar_type()), in.stride(0), ptr(ids), idx_code(ids.scalar_type()), ids.stride(0), ids.stride(1), fptr(weights),
                    weights.stride(0), weights.stride(1), ptr(index), idx_code(index.scalar_type()), index.stride(0), index.stride(1), ptr(out),
                    in_code(out.scalar_type()), out.stride(0), out.size(0), out.size(1), ids.size(1), stream);
}

bool routing_ok(const at::Tensor& ids, const at::Tensor& weights, int64_t T) {
  return idx_code(ids.scalar_type()) >= 0 && ids.dim() == 2 && ids.size(0) == T && ids.size(1) > 0 && is_f32(weights) && weights.sizes() == ids.sizes();
}

// ep_gather(input, topk_ids, topk_weight, index, output) -> True
PyObject* ep_gather(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_EXCEPTIONS_BEGIN
  const at::Tensor* t[5];
  if (n != 5 || !all_plain(args, t)) NOT_PLAIN;
  const at::Tensor &in = *t[0], &ids = *t[1], &weights = *t[2], &index = *t[3], &out = *t[4];
  if (in.dim() != 2 || out.dim() != 2 || in.numel() == 0 || out.numel() == 0 || in.size(1) != out.size(1) || out.size(1) % 8 != 0 || in.stride(1) != 1 ||
      out.stride(1) != 1 || in_code(in.scalar_type()) < 0 || in_code(out.scalar_type()) < 0 || !routing_ok(ids, weights, out.size(0)) ||
      idx_code(index.scalar_type()) < 0 || index.sizes() != ids.sizes())
    NOT_PLAIN;
  const OpRecord record("dlblas::ep_gather", t);
  DeviceScope scope(in);
  int rc;
  {
    const NoGil nogil;
    rc = gather(in, ids, weights, index, out, stream_of(in));
  }
  if (rc != DLB_OK) NOT_PLAIN;
  written(out);
  Py_RETURN_TRUE;
  HANDLE_EXCEPTIONS_END
}

// fused_moe_v3(tokens_q, tokens_scale, topk_idx, topk_weights, w13, w13_s, w2, w2_s, counts) -> combined (bf16)
PyObject* fused_moe_v3(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_EXCEPTIONS_BEGIN
  const at::Tensor* t[8];
  if (n != 9 || !all_plain(args, t) || !PyList_CheckExact(args[8])) NOT_PLAIN;
  const at::Tensor &x = *t[0], &x_s = *t[1], &ids = *t[2], &weights = *t[3], &w13 = *t[4], &w13_s = *t[5], &w2 = *t[6], &w2_s = *t[7];
  const int64_t E = PyList_GET_SIZE(args[8]);
  if (E == 0 || E > 256) NOT_PLAIN;
  int32_t counts[256];
  int64_t rows = 0, used = 0;
  for (int64_t e = 0; e < E; ++e) {
    PyObject* v = PyList_GET_ITEM(args[8], e);
    if (!PyLong_CheckExact(v)) NOT_PLAIN;
    const long long c = PyLong_AsLongLong(v);
    if (PyErr_Occurred() || c < 0 || c > (1 << 28) || c % kBlock != 0) {
      PyErr_Clear();
      NOT_PLAIN;
    }
    counts[e] = static_cast<int32_t>(c);
    rows += c;
    used += c > 0;
  }
  if (rows <= 0 || rows >= (1ll << 31) || !weights_ok(w13, w13_s) || !weights_ok(w2, w2_s)) NOT_PLAIN;
  const int64_t N = w13.size(1), H = w13.size(2), inter = N / 2;
  if (w13.size(0) != E || w2.size(0) != E || w2.size(1) != H || w2.size(2) != inter || N % (2 * kBlock) != 0 || H % kBlock != 0) NOT_PLAIN;
  if (!is_f8(x) || !is_f32(x_s) || x.dim() != 2 || x.size(1) != H || !x.is_contiguous() || x.size(0) == 0 || x_s.dim() != 2 || x_s.size(0) != x.size(0) ||
      x_s.size(1) != H / kBlock)
    NOT_PLAIN;
  const int64_t T = x.size(0), topk = ids.dim() == 2 ? ids.size(1) : 0;
  if (!routing_ok(ids, weights, T) || T * H >= (1ll << 31)) NOT_PLAIN;
  DeviceScope scope(x);
  const hipStream_t stream = stream_of(x);
  Workspace ws;
  if (!workspace_of(scope.dev, stream, x, &ws)) return nullptr;
  if (abi.scatter_ws(T, topk, E) > ws.bytes) NOT_PLAIN;
  // typical rows of an expert: half a block of its span is padding on average
  const int64_t rows_each = std::max<int64_t>(1, std::min(rows / used - 64, ceil_div(T * topk, used)));
  Form up_form, down_form;
  {
    const NoGil nogil;
    up_form = expert_form(1, rows, N, H, E, rows_each, true, ws);
    down_form = expert_form(1, rows, H, inter, E, rows_each, false, ws);
  }
  if (up_form == kStepsApart) NOT_PLAIN;
  const OpRecord record("dlblas::fused_moe_v3", t);

  at::Tensor out;
  int rc;
  bool begun = false;
  {
    const NoGil nogil;
    // one allocation for the int32 tables: expert and token of every row, row ranges and first free rows of the experts
    at::Tensor tables = empty({2 * rows + 3 * E}, at::kInt, x);
    int32_t* row_expert = iptr(tables);
    int32_t *row_token = row_expert + rows, *row_start = row_token + rows, *row_end = row_start + E, *first_free = row_end + E;
    at::Tensor slot_row = empty(ids.sizes(), ids.scalar_type(), x);
    at::Tensor q = empty({rows, inter}, at::kFloat8_e4m3fn, x);
    at::Tensor s = empty({rows, inter / kBlock}, at::kFloat, x);
    at::Tensor down = empty({rows, H}, at::kBFloat16, x);
    out = empty({T, H}, at::kBFloat16, x);
    const int32_t g = static_cast<int32_t>(E), hint = static_cast<int32_t>(rows_each);
    const Together together(ws);  // the down GEMM reads what the gate/up GEMM leaves in the workspace
    rc = abi.scatter_rows(ptr(ids), idx_code(ids.scalar_type()), ids.stride(0), ids.stride(1), counts, row_start, row_end, first_free, row_expert, row_token,
                          rows, ptr(slot_row), idx_code(slot_row.scalar_type()), topk, 1, T, topk, E, ws.ptr, ws.bytes, stream);
    // the order the down GEMM reads in place: rows whole, or the rows of a K block together
    const int64_t s_m = down_form == kOnRowRanges ? inter / kBlock : 1, s_k = down_form == kOnRowRanges ? 1 : rows;
    if (rc == DLB_OK && up_form == kOnRowRanges) {
      rc = abi.ragged_act(ptr(x), ptr(w13), fptr(x_s), fptr(w13_s), ptr(q), fptr(s), row_start, row_end, row_token, T, hint, rows, N, H, g, x_s.stride(0),
                          x_s.stride(1), s_m, s_k, 1e-10f, ws.ptr, ws.bytes, stream);
      if (rc == DLB_ERR_BAD_SHAPE) up_form = kOnWholeBlocks, rc = DLB_OK;
      begun = up_form == kOnRowRanges;
    }
    if (rc == DLB_OK && up_form == kOnWholeBlocks) {
      rc = abi.contiguous_gather_act(ptr(x), ptr(w13), fptr(x_s), fptr(w13_s), ptr(q), fptr(s), row_expert, row_token, T, rows, N, H, g, x_s.stride(0),
                                     x_s.stride(1), s_m, s_k, 1e-10f, ws.ptr, ws.bytes, stream);
      begun = rc != DLB_ERR_BAD_SHAPE;  // declined: the Python path starts over with the three steps
    }
    if (rc == DLB_OK) {
      rc = DLB_ERR_BAD_SHAPE;
      if (down_form == kOnRowRanges)
        rc = abi.ragged(ptr(q), ptr(w2), fptr(s), fptr(w2_s), ptr(down), row_start, row_end, hint, rows, H, inter, g, s_m, s_k, DLB_OUT_BF16, stream);
      if (rc == DLB_ERR_BAD_SHAPE) {
        const auto gemm = up_form == kOnWholeBlocks ? abi.contiguous_same_rows : abi.contiguous;  // the lists the gate/up GEMM left
        rc = gemm(ptr(q), ptr(w2), fptr(s), fptr(w2_s), ptr(down), row_expert, rows, H, inter, g, s_m, s_k, DLB_OUT_BF16, ws.ptr, ws.bytes, stream);
      }
    }
    if (rc == DLB_OK) rc = gather(down, ids, weights, slot_row, out, stream);
  }
  if (rc != DLB_OK) {
    if (begun) return launch_failed(rc);
    NOT_PLAIN;
  }
  return THPVariable_Wrap(std::move(out));
  HANDLE_EXCEPTIONS_END
}

// init(addresses, make_workspace): addresses in the order of Abi's members
PyObject* init(PyObject*, PyObject* args) {
  PyObject *list, *make;
  if (!PyArg_ParseTuple(args, "O!O", &PyList_Type, &list, &make)) return nullptr;
  void* slots[sizeof(Abi) / sizeof(void*)];
  if (PyList_GET_SIZE(list) != static_cast<Py_ssize_t>(sizeof(slots) / sizeof(void*)))
    return PyErr_Format(PyExc_ValueError, "%zu addresses expected", sizeof(slots) / sizeof(void*));
  for (size_t i = 0; i < sizeof(slots) / sizeof(void*); ++i) {
    slots[i] = PyLong_AsVoidPtr(PyList_GET_ITEM(list, i));
    if (!slots[i]) return PyErr_Occurred() ? nullptr : PyErr_Format(PyExc_ValueError, "address %zu is NULL", i);
  }
  memcpy(&abi, slots, sizeof(abi));
  Py_INCREF(make);
  Py_XSETREF(g_make_workspace, make);
  Py_RETURN_NONE;
}

#define FAST(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(name)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {FAST(fp8_gemm), FAST(quant), FAST(grouped_contiguous), FAST(grouped_masked), FAST(low_latency_experts), FAST(ep_gather),
                         FAST(fused_moe_v3), {"init", init, METH_VARARGS, nullptr}, {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host() { return PyModule_Create(&module); }
