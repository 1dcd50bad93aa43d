// Direct calls of the library's hot entry points from Python (module vllm_amd._fast_calls).
//
// What bounds a decode-sized call is the host: a layer's kernel takes 4 .. 20 us, while the registered op behind it
// costs the dispatcher's boxed argument matching, the host checks in Python, an allocation through the dispatcher and a
// ctypes call with two dozen arguments: 18 us of host time per W4A16 layer, 34 us per FP8 layer.  The functions below do
// the same work -- checks, allocation, launch -- in one C call.
//
// They take only the plain case: strided device tensors of the current device, nothing between the call and the device
// implementation (no tensor subclass, dispatch mode, function mode, profiler callback, functorch level or autograd
// graph), and arguments that pass every host check.  In any other case they return None without having done anything,
// and the caller goes through the registered op, which raises the error or does what the mode asks for.  The conditions
// here are therefore those of the checks in vllm_amd/_custom_ops.py, without the messages.
#include <Python.h>

#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/core/TensorBase.h>
#include <ATen/hip/EmptyTensor.h>
#include <ATen/record_function.h>
#include <c10/core/GradMode.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstdint>

#include "../../../include/vllm_amd_qlinear.h"

namespace {

using at::ScalarType;
using at::TensorBase;

PyObject* g_fp8_counters = nullptr;      // the dict (device index, stream) -> zeroed int32 counters of _custom_ops
thread_local bool t_tuned = false;       // a tuning override is in force on this thread (vllm_amd/_tuning.py)
PyObject* g_no_function = nullptr;       // torch._C._disabled_torch_function_impl
PyObject* g_function_name = nullptr;     // "__torch_function__"

// ------------------------------------------------------------------------------------------------ the plain case

// Keys a dense device tensor may carry without anything but the device implementation running.
bool plain_keys(const TensorBase& t) {
  static const c10::DispatchKeySet allowed =
      c10::DispatchKeySet({c10::DispatchKey::CUDA, c10::DispatchKey::ADInplaceOrView, c10::DispatchKey::AutogradCUDA,
                           c10::DispatchKey::AutocastCUDA});
  return (t.key_set().raw_repr() & ~allowed.raw_repr()) == 0;
}

bool plain_thread() {
  return (c10::impl::tls_local_dispatch_key_set().included_ - c10::default_included_set).empty() &&
         !c10::impl::TorchDispatchModeTLS::any_modes_set() && !at::impl::torch_function_mode_enabled() &&
         !at::hasCallbacks() && !t_tuned;
}

// Whether operators on `o` run as they are: a Tensor, a Parameter, or a subclass with torch's own disabled __torch_function__.
bool plain_type(PyObject* o) {
  return THPVariable_CheckExact(o) || _PyType_Lookup(Py_TYPE(o), g_function_name) == g_no_function;
}

// Allocation and launch run without the interpreter's lock: either can wait -- a launch for a place in a full hardware
// queue, an allocation for work that has to end before cached blocks can be given back -- and meanwhile the program's
// other threads go on, among them one that the device itself is waiting for (a host callback written in Python).
// Everything that touches a Python object comes before or after; an exception takes the lock back on its way out.
class NoGil {
 public:
  NoGil() : state_(PyEval_SaveThread()) {}
  ~NoGil() { PyEval_RestoreThread(state_); }
  NoGil(const NoGil&) = delete;
  NoGil& operator=(const NoGil&) = delete;

 private:
  PyThreadState* state_;
};

// A call in progress: which device it runs on, and whether everything seen so far was plain.
struct Call {
  bool ok = true;
  bool grad = c10::GradMode::is_enabled();
  int device = -1;

  const TensorBase* tensor(PyObject* o) {
    if (!THPVariable_Check(o) || !plain_type(o)) {
      ok = false;
      return nullptr;
    }
    const TensorBase& t = THPVariable_Unpack(o);
    if (!plain_keys(t) || !t.is_cuda() || t.layout() != c10::kStrided || (grad && t.requires_grad())) {
      ok = false;
      return nullptr;
    }
    if (device < 0) device = t.device().index();
    else if (device != t.device().index()) ok = false;
    return &t;
  }
  const TensorBase* optional(PyObject* o) { return o == Py_None ? nullptr : tensor(o); }
  bool current() const { return ok && device >= 0 && c10::hip::current_device() == device; }
};

PyObject* decline() {
  PyErr_Clear();      // (an argument of an unexpected type: the registered op names it)
  Py_RETURN_NONE;
}

int dtype_tag(ScalarType t) { return t == at::kHalf ? VAQ_F16 : t == at::kBFloat16 ? VAQ_BF16 : t == at::kFloat ? VAQ_F32 : -1; }
bool is16(ScalarType t) { return t == at::kHalf || t == at::kBFloat16; }
bool one_float(const TensorBase& t) { return t.scalar_type() == at::kFloat && t.numel() == 1; }
bool aligned16(const void* p) { return ((uintptr_t)p & 15) == 0; }

TensorBase empty(c10::IntArrayRef size, ScalarType dtype, int device) {
  return at::detail::empty_cuda(size, dtype, c10::Device(c10::kCUDA, (c10::DeviceIndex)device), std::nullopt);
}
void* stream_of(int device) { return (void*)c10::hip::getCurrentHIPStream((c10::DeviceIndex)device).stream(); }

PyObject* raise_status(int rc) {
  PyErr_SetString(rc == VAQ_ERR_UNSUPPORTED ? PyExc_NotImplementedError : PyExc_RuntimeError, vaq_last_error());
  return nullptr;
}

// Scratch sizes of recent problems: the library's answer depends on shape, format and device only, and planning a
// problem twice per call costs as much as the checks.  Direct mapped, one cache per thread.
struct Sizes {
  int64_t m = -1, n = 0, k = 0;
  int flags = 0;
  size_t c_tmp = 0, extra = 0;
};
constexpr int SIZE_SLOTS = 512;
Sizes& size_slot(Sizes (&cache)[SIZE_SLOTS], int64_t m, int64_t n, int64_t k, int flags) {
  const uint64_t h = ((uint64_t)m * 0x9e3779b97f4a7c15ull) ^ ((uint64_t)n * 0xc2b2ae3d27d4eb4full) ^ ((uint64_t)k * 0x165667b19e3779f9ull) ^ ((uint64_t)flags * 0xd6e8feb86659fd93ull);
  return cache[(h >> 40) & (SIZE_SLOTS - 1)];
}

// ------------------------------------------------------------------------------------------------ W4A16 GEMM

// b_q_type ids of the weight types, handed over by _custom_ops (they are defined by vllm_amd/scalar_type.py)
int64_t g_u4 = -1, g_u4b8 = -1, g_u8b128 = -1, g_fe4m3 = -1;

struct W4Call {
  const TensorBase *a, *c, *w, *bias, *scales, *zeros, *g_idx, *perm, *workspace;
  int64_t type, m, n, k;
  bool is_k_full;
};

// The GEMM on plain tensors; `out` is the result.  1 done, 0 not this way, -1 an exception is set.
int w4_gemm(const Call& call, const W4Call& q, int64_t lda, TensorBase& out) {
  const int bits = q.type == g_u4 || q.type == g_u4b8 ? 4 : (q.type == g_u8b128 || q.type == g_fe4m3 ? 8 : 0);
  if (bits == 0) return 0;
  const int64_t m = q.m, n = q.n, k = q.k, pack = 32 / bits;
  const ScalarType dtype = q.a->scalar_type();
  if (!is16(dtype) || k <= 0 || k % 128 != 0 || n <= 0 || n % 64 != 0 || m <= 0 || lda % 8 != 0 || !aligned16(q.a->const_data_ptr()))
    return 0;
  if (q.w->dim() != 2 || q.w->size(0) != k / 16 || q.w->size(1) != n / pack * 16 || !q.w->is_contiguous()) return 0;
  if (q.scales->dim() != 2 || q.scales->size(1) != n || !q.scales->is_contiguous() || q.scales->scalar_type() != dtype) return 0;
  if (q.workspace->scalar_type() != at::kInt) return 0;
  if (q.c && (!q.c->is_contiguous() || q.c->dim() != 2 || q.c->size(0) != m || q.c->size(1) != n || q.c->scalar_type() != dtype)) return 0;
  const int64_t groups = q.scales->size(0);
  bool act_order = false;
  if (q.g_idx && q.perm) {
    if (!q.g_idx->is_contiguous() || !q.perm->is_contiguous() || q.g_idx->dim() == 0 || q.perm->dim() == 0) return 0;
    const int64_t ng = q.g_idx->size(-1), np = q.perm->size(-1);
    if (!(ng == 0 && np == 0) && !(ng == k && np == k)) return 0;
    act_order = ng > 0;
    if (act_order && (!q.is_k_full || groups <= 1 || q.perm->scalar_type() != at::kInt)) return 0;
  }
  if (groups <= 0 || k % groups != 0) return 0;
  int64_t group_size = groups > 1 ? k / groups : -1;
  if (group_size != -1 && group_size != 32 && group_size != 64 && group_size != 128) return 0;
  if (q.bias && (q.bias->dim() != 1 || q.bias->size(0) != n || !q.bias->is_contiguous())) return 0;
  if (q.zeros && !q.zeros->is_contiguous()) return 0;
  const bool zp = q.zeros && q.zeros->dim() > 0 && q.zeros->size(-1) > 0;
  if (zp != (q.type == g_u4)) return 0;
  if (zp && (q.zeros->dim() != 2 || q.zeros->size(0) != groups || q.zeros->size(1) != n / pack)) return 0;
  if (q.type == g_fe4m3 && (act_order || (group_size != -1 && group_size != 128))) return 0;
  const int wtype = q.type == g_fe4m3 ? VAQ_WTYPE_FE4M3 : q.type == g_u8b128 ? VAQ_WTYPE_U8B128 : zp ? VAQ_WTYPE_U4 : VAQ_WTYPE_U4B8;

  static thread_local Sizes cache[SIZE_SLOTS];
  const int flags = ((call.device * 2 + (act_order ? 1 : 0)) * 4 + wtype) * 8 + (group_size == -1 ? 0 : (int)group_size / 32);
  Sizes& z = size_slot(cache, m, n, k, flags);
  if (z.m != m || z.n != n || z.k != k || z.flags != flags) {
    size_t counters = 0;
    const int rc = vaq_w4a16_gemm_workspace_of_format(m, n, k, (int)group_size, wtype, act_order, call.device, &z.c_tmp, &z.extra, &counters);
    z.m = -1;
    if (rc != VAQ_OK) return 0;
    z.m = m; z.n = n; z.k = k; z.flags = flags;
  }
  int rc;
  {
    NoGil nogil;
    if (q.c) out = *q.c;
    else out = empty({m, n}, dtype, call.device);
    TensorBase c_tmp, a_tmp;
    if (z.c_tmp) c_tmp = empty({(int64_t)(z.c_tmp / 4)}, at::kFloat, call.device);
    if (z.extra) a_tmp = empty({(int64_t)(z.extra / 2)}, dtype, call.device);
    rc = vaq_w4a16_gemm(
        q.a->const_data_ptr(), lda, (const int32_t*)q.w->const_data_ptr(), q.scales->const_data_ptr(),
        zp ? (const int32_t*)q.zeros->const_data_ptr() : nullptr, act_order ? (const int32_t*)q.perm->const_data_ptr() : nullptr,
        q.bias ? q.bias->const_data_ptr() : nullptr, out.mutable_data_ptr(), z.c_tmp ? (float*)c_tmp.mutable_data_ptr() : nullptr,
        (int64_t)z.c_tmp, z.extra ? a_tmp.mutable_data_ptr() : nullptr, (int32_t*)q.workspace->mutable_data_ptr(),
        q.workspace->numel(), m, n, k, (int)group_size, dtype_tag(dtype), wtype, 0, stream_of(call.device));
  }
  if (rc != VAQ_OK) {
    raise_status(rc);
    return -1;
  }
  return 1;
}

// w4_gemm(a, c, w, bias, scales, zeros, g_idx, perm, workspace, type_id, m, n, k, is_k_full) -> Tensor | None
PyObject* py_w4_gemm(PyObject*, PyObject* const* v, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  if (nargs != 14 || !plain_thread()) return decline();
  Call call;
  W4Call q;
  q.a = call.tensor(v[0]);
  q.c = call.optional(v[1]);
  q.w = call.tensor(v[2]);
  q.bias = call.optional(v[3]);
  q.scales = call.tensor(v[4]);
  q.zeros = call.optional(v[5]);
  q.g_idx = call.optional(v[6]);
  q.perm = call.optional(v[7]);
  q.workspace = call.tensor(v[8]);
  if (!call.current()) return decline();
  q.type = PyLong_AsLongLong(v[9]);
  q.m = PyLong_AsLongLong(v[10]);
  q.n = PyLong_AsLongLong(v[11]);
  q.k = PyLong_AsLongLong(v[12]);
  q.is_k_full = v[13] == Py_True;
  if (PyErr_Occurred()) return decline();
  if (q.a->dim() != 2 || q.a->size(0) != q.m || q.a->size(1) != q.k || q.a->stride(1) != 1) return decline();
  TensorBase out;
  const int r = w4_gemm(call, q, q.a->stride(0), out);
  if (r < 0) return nullptr;
  if (r == 0) return decline();
  if (q.c) return Py_NewRef(v[1]);
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// The activations of a linear layer, [..., k]: rows and row stride of the matrix they are, without making a view of them.
bool as_rows(const TensorBase& x, int64_t k, int64_t* rows, int64_t* ld) {
  const int64_t d = x.dim();
  if (d < 1 || x.size(d - 1) != k || (x.stride(d - 1) != 1)) return false;
  if (d == 2) {
    *rows = x.size(0);
    *ld = x.stride(0);
    return true;
  }
  if (!x.is_contiguous()) return false;
  *rows = x.numel() / k;
  *ld = k;
  return true;
}

// The result [rows, n] as the layer returns it, [..., n].
PyObject* wrap_rows(const TensorBase& x, TensorBase out, int64_t n) {
  if (x.dim() != 2) {
    c10::SmallVector<int64_t, 6> size(x.sizes().begin(), x.sizes().end());
    c10::SmallVector<int64_t, 6> stride(size.size());
    size.back() = n;
    int64_t s = 1;
    for (size_t i = size.size(); i-- > 0; s *= size[i]) stride[i] = s;
    out.unsafeGetTensorImpl()->set_sizes_and_strides(size, stride);      // (fresh and contiguous: its own storage, no other view)
  }
  return THPVariable_Wrap(std::move(out));
}

// w4_linear(x, w, bias, scales, zeros, g_idx, perm, workspace, type_id, n, k, is_k_full) -> Tensor [..., n] | None
PyObject* py_w4_linear(PyObject*, PyObject* const* v, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  if (nargs != 12 || !plain_thread()) return decline();
  Call call;
  W4Call q;
  q.a = call.tensor(v[0]);
  q.c = nullptr;
  q.w = call.tensor(v[1]);
  q.bias = call.optional(v[2]);
  q.scales = call.tensor(v[3]);
  q.zeros = call.optional(v[4]);
  q.g_idx = call.optional(v[5]);
  q.perm = call.optional(v[6]);
  q.workspace = call.tensor(v[7]);
  if (!call.current()) return decline();
  q.type = PyLong_AsLongLong(v[8]);
  q.n = PyLong_AsLongLong(v[9]);
  q.k = PyLong_AsLongLong(v[10]);
  q.is_k_full = v[11] == Py_True;
  if (PyErr_Occurred()) return decline();
  int64_t lda = 0;
  if (q.k <= 0 || !as_rows(*q.a, q.k, &q.m, &lda)) return decline();
  TensorBase out;
  const int r = w4_gemm(call, q, lda, out);
  if (r < 0) return nullptr;
  if (r == 0) return decline();
  return wrap_rows(*q.a, std::move(out), q.n);
  END_HANDLE_TH_ERRORS
}

// ------------------------------------------------------------------------------------------------ FP8

// The weight, scales and bias of an FP8 GEMM against K columns of activations in `out_type`.
bool fp8_weight_ok(const TensorBase& b, const TensorBase& sb, const TensorBase* bias, int64_t k, ScalarType out_type) {
  if (b.scalar_type() != at::kFloat8_e4m3fn || b.dim() != 2 || b.size(0) != k || b.stride(0) != 1 || b.stride(1) % 16 != 0) return false;
  const int64_t n = b.size(1);
  if (k <= 0 || n <= 0 || k % 16 != 0 || n % 16 != 0 || !is16(out_type)) return false;
  if (sb.scalar_type() != at::kFloat || !sb.is_contiguous() || (sb.numel() != 1 && sb.numel() != n)) return false;
  return !bias || (bias->dim() == 1 && bias->numel() == n && bias->is_contiguous() && bias->scalar_type() == out_type);
}

// What one GEMM needs for its K split, found before anything is launched.  1 ready, 0 not this way, -1 an exception is set.
struct Fp8Scratch {
  size_t c_tmp_bytes = 0;
  TensorBase counters;      // (a reference of its own: the table of counters may change while the lock is given up)
  void* stream = nullptr;
};
int fp8_scratch(const Call& call, int64_t m, int64_t n, int64_t k, Fp8Scratch& s) {
  static thread_local Sizes cache[SIZE_SLOTS];
  Sizes& z = size_slot(cache, m, n, k, call.device);
  if (z.m != m || z.n != n || z.k != k || z.flags != call.device) {
    z.m = -1;
    if (vaq_fp8_scaled_mm_workspace(m, n, k, &z.c_tmp, &z.extra) != VAQ_OK) return 0;
    z.m = m; z.n = n; z.k = k; z.flags = call.device;
  }
  s.stream = stream_of(call.device);
  s.c_tmp_bytes = z.c_tmp;
  if (!z.c_tmp) return 1;
  // arrival counters: one zeroed array per device and stream, kept by _custom_ops (which makes it on a stream's first call)
  PyObject* key = Py_BuildValue("(iK)", call.device, (unsigned long long)(uintptr_t)s.stream);
  if (!key) return -1;
  PyObject* t = PyDict_GetItemWithError(g_fp8_counters, key);      // borrowed
  Py_DECREF(key);
  if (!t || !THPVariable_Check(t)) return PyErr_Occurred() ? -1 : 0;
  const TensorBase& c = THPVariable_Unpack(t);
  if (c.numel() < (int64_t)z.extra) return 0;
  s.counters = c;
  return 1;
}

// (without the lock)
int fp8_mm(const Fp8Scratch& s, const void* a, int64_t lda, int64_t m, const float* sa, int64_t sa_count, const TensorBase& b,
           const TensorBase& sb, const TensorBase* bias, const TensorBase& out) {
  const int64_t k = b.size(0), n = b.size(1);
  TensorBase c_tmp;
  if (s.c_tmp_bytes) c_tmp = empty({(int64_t)(s.c_tmp_bytes / 4)}, at::kFloat, out.device().index());
  return vaq_fp8_scaled_mm_ws((const uint8_t*)a, lda, (const uint8_t*)b.const_data_ptr(), b.stride(1), sa, sa_count,
                              (const float*)sb.const_data_ptr(), sb.numel(), bias ? bias->const_data_ptr() : nullptr,
                              out.mutable_data_ptr(), n, dtype_tag(out.scalar_type()), m, n, k,
                              s.c_tmp_bytes ? (float*)c_tmp.mutable_data_ptr() : nullptr, (int64_t)s.c_tmp_bytes,
                              s.c_tmp_bytes ? (int32_t*)s.counters.mutable_data_ptr() : nullptr,
                              s.c_tmp_bytes ? s.counters.numel() : 0, s.stream);
}

// scaled_mm(a, b, scale_a, scale_b, out_dtype, bias) -> Tensor [..., n] | None
PyObject* py_scaled_mm(PyObject*, PyObject* const* v, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  if (nargs != 6 || !plain_thread() || !THPDtype_Check(v[4])) return decline();
  Call call;
  const TensorBase* a = call.tensor(v[0]);
  const TensorBase* b = call.tensor(v[1]);
  const TensorBase* sa = call.tensor(v[2]);
  const TensorBase* sb = call.tensor(v[3]);
  const TensorBase* bias = call.optional(v[5]);
  if (!call.current()) return decline();
  const ScalarType out_type = ((THPDtype*)v[4])->scalar_type;
  if (b->dim() != 2 || a->scalar_type() != at::kFloat8_e4m3fn || !fp8_weight_ok(*b, *sb, bias, b->size(0), out_type)) return decline();
  int64_t m = 0, lda = 0;
  if (!as_rows(*a, b->size(0), &m, &lda) || m <= 0 || lda % 16 != 0) return decline();
  if (sa->scalar_type() != at::kFloat || !sa->is_contiguous() || (sa->numel() != 1 && sa->numel() != m)) return decline();
  Fp8Scratch scratch;
  const int r = fp8_scratch(call, m, b->size(1), b->size(0), scratch);
  if (r < 0) return nullptr;
  if (r == 0) return decline();
  TensorBase out;
  int rc;
  {
    NoGil nogil;
    out = empty({m, b->size(1)}, out_type, call.device);
    rc = fp8_mm(scratch, a->const_data_ptr(), lda, m, (const float*)sa->const_data_ptr(), sa->numel(), *b, *sb, bias, out);
  }
  if (rc != VAQ_OK) return raise_status(rc);
  return wrap_rows(*a, std::move(out), b->size(1));
  END_HANDLE_TH_ERRORS
}

// fp8_linear(x, weight, weight_scale, input_scale or None, scale_ub or None, out_dtype, bias) -> Tensor [..., n] | None
// Activations quantised per token (input_scale None) or with a static per-tensor scale, then the GEMM: one launch for a few
// rows, else two, and the quantised activations and their scales are one allocation that nobody else sees.
PyObject* py_fp8_linear(PyObject*, PyObject* const* v, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  if (nargs != 7 || !plain_thread() || !THPDtype_Check(v[5])) return decline();
  Call call;
  const TensorBase* x = call.tensor(v[0]);
  const TensorBase* b = call.tensor(v[1]);
  const TensorBase* sb = call.tensor(v[2]);
  const TensorBase* in_scale = call.optional(v[3]);
  const TensorBase* ub = call.optional(v[4]);
  const TensorBase* bias = call.optional(v[6]);
  if (!call.current()) return decline();
  const ScalarType out_type = ((THPDtype*)v[5])->scalar_type;
  const int in_tag = dtype_tag(x->scalar_type());
  if (in_tag < 0 || b->dim() != 2 || !fp8_weight_ok(*b, *sb, bias, b->size(0), out_type)) return decline();
  if ((in_scale && (!one_float(*in_scale) || ub)) || (ub && !one_float(*ub))) return decline();
  const int64_t k = b->size(0), n = b->size(1);
  int64_t m = 0, ldx = 0;
  if (!as_rows(*x, k, &m, &ldx) || m <= 0) return decline();
  TensorBase out;
  int rc;
  // a few rows: one launch that quantises what it multiplies, unless the strides are beyond it
  const bool x_ok = x->scalar_type() == out_type && ldx >= k && ldx % 8 == 0 && aligned16(x->const_data_ptr());
  if (!ub && x_ok && vaq_fp8_quant_scaled_mm_takes(m, n, k, in_scale == nullptr)) {
    {
      NoGil nogil;
      out = empty({m, n}, out_type, call.device);
      rc = vaq_fp8_quant_scaled_mm(x->const_data_ptr(), ldx, in_scale ? (const float*)in_scale->const_data_ptr() : nullptr,
                                   (const uint8_t*)b->const_data_ptr(), b->stride(1), (const float*)sb->const_data_ptr(),
                                   sb->numel(), bias ? bias->const_data_ptr() : nullptr, out.mutable_data_ptr(), n, in_tag, m,
                                   n, k, stream_of(call.device));
    }
    if (rc == VAQ_OK) return wrap_rows(*x, std::move(out), n);
    if (rc != VAQ_ERR_UNSUPPORTED) return raise_status(rc);
  }
  Fp8Scratch scratch;
  const int r = fp8_scratch(call, m, n, k, scratch);
  if (r < 0) return nullptr;
  if (r == 0) return decline();
  {
    NoGil nogil;
    const int64_t codes = m * k;      // (a multiple of 16: the scales behind them are aligned)
    TensorBase q = empty({codes + (in_scale ? 0 : 4 * m)}, at::kByte, call.device);
    uint8_t* qp = (uint8_t*)q.mutable_data_ptr();
    const float* sa = in_scale ? (const float*)in_scale->const_data_ptr() : (const float*)(qp + codes);
    out = empty({m, n}, out_type, call.device);
    rc = in_scale ? vaq_fp8_quant_static(x->const_data_ptr(), in_tag, ldx, qp, k, sa, m, k, scratch.stream)
                  : vaq_fp8_quant_per_token(x->const_data_ptr(), in_tag, ldx, qp, k, (float*)(qp + codes),
                                            ub ? (const float*)ub->const_data_ptr() : nullptr, m, k, scratch.stream);
    if (rc == VAQ_OK) rc = fp8_mm(scratch, qp, k, m, sa, in_scale ? 1 : m, *b, *sb, bias, out);
  }
  if (rc != VAQ_OK) return raise_status(rc);
  return wrap_rows(*x, std::move(out), n);
  END_HANDLE_TH_ERRORS
}

// fp8_quant(input, scale or None, scale_ub or None, per_token, output or None) -> (output, scale) | None
// The output of a static or per-token quantisation of [tokens, hidden]; dynamic per tensor and padded outputs go through
// the registered op.
PyObject* py_fp8_quant(PyObject*, PyObject* const* v, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  if (nargs != 5 || !plain_thread()) return decline();
  Call call;
  const TensorBase* x = call.tensor(v[0]);
  const TensorBase* scale = call.optional(v[1]);
  const TensorBase* ub = call.optional(v[2]);
  const TensorBase* given = call.optional(v[4]);
  if (!call.current()) return decline();
  if (!scale && v[3] != Py_True) return decline();
  const int in_tag = dtype_tag(x->scalar_type());
  if (in_tag < 0 || x->dim() != 2 || x->stride(1) != 1 || x->size(0) <= 0 || x->size(1) <= 0) return decline();
  const int64_t m = x->size(0), k = x->size(1);
  if (given && (given->scalar_type() != at::kFloat8_e4m3fn || given->dim() != 2 || given->size(0) != m || given->size(1) != k ||
                given->stride(1) != 1))
    return decline();
  if ((scale && !one_float(*scale)) || (ub && !one_float(*ub))) return decline();
  TensorBase out, scales;
  int rc;
  {
    NoGil nogil;
    out = given ? *given : empty({m, k}, at::kFloat8_e4m3fn, call.device);
    void* stream = stream_of(call.device);
    if (scale) {
      rc = vaq_fp8_quant_static(x->const_data_ptr(), in_tag, x->stride(0), (uint8_t*)out.mutable_data_ptr(), out.stride(0),
                                (const float*)scale->const_data_ptr(), m, k, stream);
    } else {
      scales = empty({m, 1}, at::kFloat, call.device);
      rc = vaq_fp8_quant_per_token(x->const_data_ptr(), in_tag, x->stride(0), (uint8_t*)out.mutable_data_ptr(), out.stride(0),
                                   (float*)scales.mutable_data_ptr(), ub ? (const float*)ub->const_data_ptr() : nullptr, m, k, stream);
    }
  }
  if (rc != VAQ_OK) return raise_status(rc);
  return Py_BuildValue("(NN)", given ? Py_NewRef(v[4]) : THPVariable_Wrap(std::move(out)),
                       scale ? Py_NewRef(v[1]) : THPVariable_Wrap(std::move(scales)));
  END_HANDLE_TH_ERRORS
}

// The operands every norm operator shares: input [..., hidden] whose rows lie one stride apart, weight, residual.
bool norm_ok(const TensorBase& in, const TensorBase& weight, const TensorBase* residual, int64_t* tokens, int64_t* stride) {
  const int64_t d = in.dim();
  if (d < 1 || !is16(in.scalar_type()) || in.size(d - 1) <= 0 || !as_rows(in, in.size(d - 1), tokens, stride) || *tokens <= 0) return false;
  if (weight.scalar_type() != in.scalar_type() || weight.numel() != in.size(d - 1) || !weight.is_contiguous()) return false;
  return !residual || (residual->scalar_type() == in.scalar_type() && residual->is_contiguous() && residual->sizes() == in.sizes());
}

// rms_norm_dynamic_quant(input, weight, epsilon, scale_ub or None, residual or None) -> (output, scales [tokens, 1]) | None
PyObject* py_rms_norm_dynamic_quant(PyObject*, PyObject* const* v, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  if (nargs != 5 || !plain_thread()) return decline();
  Call call;
  const TensorBase* x = call.tensor(v[0]);
  const TensorBase* weight = call.tensor(v[1]);
  const TensorBase* ub = call.optional(v[3]);
  const TensorBase* residual = call.optional(v[4]);
  if (!call.current()) return decline();
  const double eps = PyFloat_AsDouble(v[2]);
  int64_t tokens = 0, stride = 0;
  if (PyErr_Occurred() || !norm_ok(*x, *weight, residual, &tokens, &stride) || (ub && !one_float(*ub))) return decline();
  // (the output takes the memory format of the input: the rows of a strided one are left to the registered op)
  if (!x->is_contiguous()) return decline();
  TensorBase out, scales;
  int rc;
  {
    NoGil nogil;
    out = empty(x->sizes(), at::kFloat8_e4m3fn, call.device);
    scales = empty({tokens, 1}, at::kFloat, call.device);
    rc = vaq_rms_norm_dynamic_per_token_fp8_quant(
        (uint8_t*)out.mutable_data_ptr(), (float*)scales.mutable_data_ptr(), x->const_data_ptr(), stride, weight->const_data_ptr(),
        ub ? (const float*)ub->const_data_ptr() : nullptr, (float)eps, residual ? residual->mutable_data_ptr() : nullptr,
        dtype_tag(x->scalar_type()), tokens, x->size(-1), stream_of(call.device));
  }
  if (rc != VAQ_OK) return raise_status(rc);
  return Py_BuildValue("(NN)", THPVariable_Wrap(std::move(out)), THPVariable_Wrap(std::move(scales)));
  END_HANDLE_TH_ERRORS
}

// rms_norm_static_quant(out, input, residual or None, weight, scale, epsilon) -> True | None
PyObject* py_rms_norm_static_quant(PyObject*, PyObject* const* v, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  if (nargs != 6 || !plain_thread()) return decline();
  Call call;
  const TensorBase* out = call.tensor(v[0]);
  const TensorBase* x = call.tensor(v[1]);
  const TensorBase* residual = call.optional(v[2]);
  const TensorBase* weight = call.tensor(v[3]);
  const TensorBase* scale = call.tensor(v[4]);
  if (!call.current()) return decline();
  const double eps = PyFloat_AsDouble(v[5]);
  int64_t tokens = 0, stride = 0;
  if (PyErr_Occurred() || !norm_ok(*x, *weight, residual, &tokens, &stride) || !one_float(*scale) ||
      out->scalar_type() != at::kFloat8_e4m3fn || !out->is_contiguous() || out->numel() != x->numel())
    return decline();
  int rc;
  {
    NoGil nogil;
    rc = vaq_rms_norm_static_fp8_quant((uint8_t*)out->mutable_data_ptr(), x->const_data_ptr(), stride, weight->const_data_ptr(),
                                       (const float*)scale->const_data_ptr(), (float)eps,
                                       residual ? residual->mutable_data_ptr() : nullptr, dtype_tag(x->scalar_type()),
                                       tokens, x->size(-1), stream_of(call.device));
  }
  if (rc != VAQ_OK) return raise_status(rc);
  Py_RETURN_TRUE;
  END_HANDLE_TH_ERRORS
}

// silu_and_mul_quant(out, input, scale) -> True | None
PyObject* py_silu_and_mul_quant(PyObject*, PyObject* const* v, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  if (nargs != 3 || !plain_thread()) return decline();
  Call call;
  const TensorBase* out = call.tensor(v[0]);
  const TensorBase* x = call.tensor(v[1]);
  const TensorBase* scale = call.tensor(v[2]);
  if (!call.current()) return decline();
  if (out->scalar_type() != at::kFloat8_e4m3fn || !is16(x->scalar_type()) || x->dim() < 1 || x->size(-1) <= 0 || x->size(-1) % 2 != 0 ||
      !one_float(*scale) || !x->is_contiguous() || !out->is_contiguous())
    return decline();
  const int64_t d = x->size(-1) / 2, tokens = x->numel() / (2 * d);
  if (tokens <= 0 || out->numel() != tokens * d) return decline();
  int rc;
  {
    NoGil nogil;
    rc = vaq_silu_and_mul_fp8_quant((uint8_t*)out->mutable_data_ptr(), x->const_data_ptr(), (const float*)scale->const_data_ptr(),
                                    dtype_tag(x->scalar_type()), tokens, d, stream_of(call.device));
  }
  if (rc != VAQ_OK) return raise_status(rc);
  Py_RETURN_TRUE;
  END_HANDLE_TH_ERRORS
}

// repack(codes, perm or None, k, n, bits, layout) -> Tensor | None; perm None: an AWQ checkpoint's tensor
PyObject* py_repack(PyObject*, PyObject* const* v, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  if (nargs != 6 || !plain_thread()) return decline();
  Call call;
  const TensorBase* w = call.tensor(v[0]);
  const TensorBase* perm = call.optional(v[1]);
  if (!call.current()) return decline();
  const int64_t k = PyLong_AsLongLong(v[2]), n = PyLong_AsLongLong(v[3]), bits = PyLong_AsLongLong(v[4]), layout = PyLong_AsLongLong(v[5]);
  if (PyErr_Occurred() || k <= 0 || n <= 0 || k % 16 != 0 || n % 64 != 0 || (bits != 4 && bits != 8) || (!perm && bits != 4)) return decline();
  const int64_t pack = 32 / bits;
  if (w->scalar_type() != at::kInt || !w->is_contiguous() || w->dim() != 2 || w->size(0) != (perm ? k / pack : k) ||
      w->size(1) != (perm ? n : n / pack))
    return decline();
  if (perm && (perm->scalar_type() != at::kInt || !perm->is_contiguous() || (perm->numel() != 0 && perm->numel() != k))) return decline();
  TensorBase out;
  int rc;
  {
    NoGil nogil;
    out = empty({k / 16, n * 16 / pack}, at::kInt, call.device);
    const int32_t* src = (const int32_t*)w->const_data_ptr();
    int32_t* dst = (int32_t*)out.mutable_data_ptr();
    rc = perm ? vaq_w4a16_repack(src, perm->numel() ? (const int32_t*)perm->const_data_ptr() : nullptr, dst, k, n, (int)bits,
                                 (int)layout, stream_of(call.device))
              : vaq_w4a16_repack_awq(src, dst, k, n, (int)bits, (int)layout, stream_of(call.device));
  }
  if (rc != VAQ_OK) return raise_status(rc);
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// tuned(on) -> what it was: whether this thread's calls are left to the registered ops, which pass the override on
PyObject* py_tuned(PyObject*, PyObject* on) {
  const int value = PyObject_IsTrue(on);
  if (value < 0) return nullptr;
  const bool was = t_tuned;
  t_tuned = value != 0;
  return PyBool_FromLong(was);
}

// setup(fp8_counters: dict, (u4, u4b8, u8b128, fe4m3): ids)
PyObject* py_setup(PyObject*, PyObject* args) {
  PyObject* counters;
  long long u4, u4b8, u8b128, fe4m3;
  if (!PyArg_ParseTuple(args, "O!(LLLL)", &PyDict_Type, &counters, &u4, &u4b8, &u8b128, &fe4m3)) return nullptr;
  Py_XSETREF(g_fp8_counters, Py_NewRef(counters));
  if (!g_no_function) {
    PyObject* torch_c = PyImport_ImportModule("torch._C");
    if (!torch_c) return nullptr;
    g_no_function = PyObject_GetAttrString(torch_c, "_disabled_torch_function_impl");
    Py_DECREF(torch_c);
    g_function_name = PyUnicode_InternFromString("__torch_function__");
    if (!g_no_function || !g_function_name) return nullptr;
  }
  g_u4 = u4; g_u4b8 = u4b8; g_u8b128 = u8b128; g_fe4m3 = fe4m3;
  Py_RETURN_NONE;
}

#define FAST(name) {#name, (PyCFunction)(void (*)(void))py_##name, METH_FASTCALL, nullptr}
PyMethodDef g_methods[] = {
    {"setup", py_setup, METH_VARARGS, nullptr},
    {"tuned", py_tuned, METH_O, nullptr},
    FAST(w4_gemm), FAST(w4_linear), FAST(scaled_mm), FAST(fp8_linear), FAST(fp8_quant), FAST(rms_norm_dynamic_quant),
    FAST(rms_norm_static_quant), FAST(silu_and_mul_quant), FAST(repack), {nullptr, nullptr, 0, nullptr}};
PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_fast_calls", nullptr, -1, g_methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__fast_calls(void) { return PyModule_Create(&g_module); }
