// The host path in native code: what a call of a quantized Linear, or of a whole fused decoder block, does between
// Python and the C ABI -- reading the modules' tensors, checking them, allocating outputs and queueing the launches.
//
// Why it exists: the decode kernels run for 4 to 9 us, and a launch costs the host 2.4 us, but the same call made
// from Python through ctypes took 19 us (argument conversion, a workspace lookup by stream, three tensor
// allocations through the dispatcher, a device context); a block's decode step of six launches took 114 us against
// 43 us of kernels, and the 24-layer model's 2.45 ms against 0.75 ms.
//
// Every function here serves the plain case only: tensors of exactly torch.Tensor or nn.Parameter, contiguous, on the
// current device, of the types the kernels take.  For anything else it returns None (nothing has been queued then) and
// the Python code that calls it goes on with its general path, which copies what is not contiguous and raises the
// errors.  So there is no second set of error messages here; what the C ABI itself refuses is raised as _abi.check does,
// and what torch throws (out of memory) as torch's own functions raise it.
#include <ATen/core/Tensor.h>
#include <ATen/hip/EmptyTensor.h>
#include <Python.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <dlfcn.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/DynamicTypes.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cmath>
#include <initializer_list>

#include "../../include/astrai_q.h"

namespace {

// ---- the C ABI, bound to whichever library _abi.load() has (the product, or the lab build in tests) -------------
#define AQ_HOST_SYMBOLS(X)                                                                                       \
  X(aq_error_string)                                                                                             \
  X(aq_quant_rowwise_i8)                                                                                         \
  X(aq_rmsnorm_quant_rowwise_i8)                                                                                 \
  X(aq_swiglu_quant_rowwise_i8)                                                                                  \
  X(aq_quant_tensor_fp8)                                                                                         \
  X(aq_quant_tensor_fp8_onepass)                                                                                 \
  X(aq_linear_w8a8_residual)                                                                                     \
  X(aq_linear_fp8_residual)                                                                                      \
  X(aq_gemv_w8a8_workspace_bytes)                                                                                \
  X(aq_gemv_w8a8_decode_one_launch)                                                                              \
  X(aq_gemv_fp8_decode_one_launch)                                                                               \
  X(aq_linear_codes_pitch)                                                                                       \
  X(aq_quant_rowwise_i8_strided)                                                                                 \
  X(aq_quant_tensor_fp8_strided)                                                                                 \
  X(aq_linear_w8a8_strided)                                                                                      \
  X(aq_linear_fp8_strided)                                                                                       \
  X(aq_linear_few_rows_ok)                                                                                       \
  X(aq_linear_few_rows_queued_ok)                                                                                \
  X(aq_linear_few_rows)                                                                                          \
  X(aq_gemv_w8a8_decode_residual)                                                                                \
  X(aq_gemv_w8a8_decode_rmsnorm)                                                                                 \
  X(aq_gemv_w8a8_codes_residual)                                                                                 \
  X(aq_gemv_w8a8_decode_swiglu_ok)                                                                               \
  X(aq_gemv_w8a8_decode_swiglu)                                                                                  \
  X(aq_gemv_w8a8_decode_attn)                                                                                    \
  X(aq_gemv_fp8_workspace_bytes)                                                                                 \
  X(aq_gemv_fp8_decode_residual)                                                                                 \
  X(aq_rope_kv_write)                                                                                            \
  X(aq_rope_kv_write_qknorm)                                                                                     \
  X(aq_rope_kv_cache_write)                                                                                      \
  X(aq_rope_paged_attn_decode)                                                                                   \
  X(aq_rope_paged_attn_decode_qknorm)                                                                            \
  X(aq_rope_paged_attn_decode_partials)                                                                          \
  X(aq_rope_paged_attn_decode_partials_qknorm)                                                                   \
  X(aq_paged_attn_decode_slices)                                                                                 \
  X(aq_paged_attn_decode_partials_bytes)                                                                         \
  X(aq_paged_attn_decode_workspace_bytes)                                                                        \
  X(aq_prefill_attn_causal_ahead)                                                                                \
  X(aq_prefill_attn_paged_ahead)                                                                                 \
  X(aq_rope_prefill_attn_causal_ahead)                                                                           \
  X(aq_rope_prefill_attn_paged_ahead)

struct Library {
#define X(name) decltype(&::name) name = nullptr;
  AQ_HOST_SYMBOLS(X)
#undef X
};
Library lib;

PyObject* none() { Py_RETURN_NONE; }

// _abi.check: what the library refused as ValueError, anything else as RuntimeError.
PyObject* fail(int code, const char* what) {
  PyObject* kind = code == AQ_E_SHAPE || code == AQ_E_DTYPE || code == AQ_E_ALIGN || code == AQ_E_RANGE ? PyExc_ValueError
                                                                                                          : PyExc_RuntimeError;
  return PyErr_Format(kind, "%s: %s (code %d)", what, lib.aq_error_string(code), code);
}

// ---- tensors ----------------------------------------------------------------------------------------------------
using at::ScalarType;
using at::Tensor;

// The tensor behind a Python object, or null: a subclass (fake, functional, quantised by someone else) is not plain.
const Tensor* unpack(PyObject* o) { return o && THPVariable_CheckExact(o) ? &THPVariable_Unpack(o) : nullptr; }

struct Held {  // a reference to a Python object (two copies of a Tensor cost 0.08 us, of its Python object nothing)
  PyObject* const o;
  explicit Held(PyObject* p) : o(p) { Py_INCREF(o); }
  ~Held() { Py_DECREF(o); }
  Held(const Held&) = delete;
};

// aq dtype code of an activation type, -1 for one the kernels do not take
int act_code(ScalarType t) { return t == ScalarType::BFloat16 ? AQ_BF16 : t == ScalarType::Float ? AQ_F32 : -1; }

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

bool plain(const Tensor& t, ScalarType type, int dev) {
  return t.is_cuda() && t.get_device() == dev && t.scalar_type() == type && t.is_contiguous();
}

struct Call {  // the device and stream of one call
  int dev = -1;
  void* stream = nullptr;
  // false: x is not on the current device (the caller's general path switches devices)
  bool at(const Tensor& x) {
    if (!x.is_cuda()) return false;
    dev = x.get_device();
    return dev == c10::hip::current_device();
  }
  void current_stream() { stream = c10::hip::getCurrentHIPStream(static_cast<c10::DeviceIndex>(dev)).stream(); }
  bool captured() const {  // (the null stream cannot be)
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    if (stream && hipStreamIsCapturing(static_cast<hipStream_t>(stream), &status) != hipSuccess) (void)hipGetLastError();
    return status != hipStreamCaptureStatusNone;
  }
  Tensor empty(at::IntArrayRef size, ScalarType type) const {
    return at::detail::empty_cuda(size, type, c10::Device(c10::kCUDA, static_cast<c10::DeviceIndex>(dev)), std::nullopt);
  }
};

struct Rows {  // x [..., K] seen as M rows
  int64_t M = 0, K = 0;
  const void* p = nullptr;
  int code = -1;
};
bool rows_of(const Tensor& x, Rows* r) {
  r->code = act_code(x.scalar_type());
  if (r->code < 0 || x.dim() < 1 || !x.is_contiguous()) return false;
  r->K = x.size(x.dim() - 1);
  if (r->K <= 0 || r->K % 16) return false;
  r->M = x.numel() / r->K;
  r->p = x.const_data_ptr();
  return r->M > 0 && aligned16(r->p);
}

struct Bias {
  Tensor hold;
  const void* p = nullptr;
  int code = 0;
};
// None, or a vector of N floats
bool bias_of(PyObject* o, int64_t N, int dev, Bias* b) {
  if (!o || o == Py_None) return true;
  const Tensor* t = unpack(o);
  if (!t || !t->is_cuda() || t->get_device() != dev || t->dim() != 1 || t->size(0) != N || !t->is_contiguous()) return false;
  b->code = act_code(t->scalar_type());
  if (b->code < 0) return false;
  b->hold = *t;
  b->p = t->const_data_ptr();
  return true;
}

// None, or M x N elements of the output's type whose last dimension is N
bool residual_of(PyObject* o, int64_t M, int64_t N, ScalarType type, int dev, const void** p) {
  *p = nullptr;
  if (!o || o == Py_None) return true;
  const Tensor* t = unpack(o);
  if (!t || !plain(*t, type, dev) || t->numel() != M * N || t->dim() < 1 || t->size(t->dim() - 1) != N) return false;
  *p = t->const_data_ptr();
  return aligned16(*p);
}

// weight codes [N, K] and scales: one per row (int8), or one for the tensor (fp8)
bool weight_of(PyObject* wq, PyObject* sw, int64_t K, int dev, bool fp8, const Tensor** w, const Tensor** s) {
  *w = unpack(wq);
  *s = unpack(sw);
  if (!*w || !*s || !plain(**w, fp8 ? ScalarType::Byte : ScalarType::Char, dev) || !plain(**s, ScalarType::Float, dev)) return false;
  if ((*w)->dim() != 2 || (*w)->size(1) != K || (*w)->size(0) < 1) return false;
  return (*s)->numel() == (fp8 ? 1 : (*w)->size(0)) && aligned16((*w)->const_data_ptr());
}

// an output type given as torch.dtype, or None for the activations'
bool out_type(PyObject* o, ScalarType like, ScalarType* t) {
  if (o == Py_None) {
    *t = like;
  } else if (THPDtype_Check(o)) {
    *t = reinterpret_cast<THPDtype*>(o)->scalar_type;
  } else {
    return false;
  }
  return act_code(*t) >= 0;
}

PyObject* pair(const Tensor& a, const Tensor& b) {
  PyObject* pa = THPVariable_Wrap(a);
  PyObject* pb = pa ? THPVariable_Wrap(b) : nullptr;
  PyObject* r = pb ? PyTuple_Pack(2, pa, pb) : nullptr;
  Py_XDECREF(pa);
  Py_XDECREF(pb);
  return r;
}

// The library calls queue work and may wait while the device's queue is full: other Python threads run meanwhile.
// The lock is taken back on every way out: an exception is turned into a Python error, which needs it.  (Not in a
// destructor: Python ends a thread that waits for the lock at exit by unwinding it from there.)
template <class F>
int queued(F&& launch) {
  PyThreadState* const thread = PyEval_SaveThread();
  int rc;
  try {
    rc = launch();
  } catch (...) {
    PyEval_RestoreThread(thread);
    throw;
  }
  PyEval_RestoreThread(thread);
  return rc;
}

#define AQ_ARGS(n)                                                                       \
  if (nargs != (n)) return PyErr_Format(PyExc_TypeError, "expected %d arguments", n);    \
  if (!lib.aq_error_string) return PyErr_Format(PyExc_RuntimeError, "no library is bound")

// ---- operators (positional arguments only; the wrappers in ops.py document them) ----------------------------------

// quant_rowwise_i8(x) -> (codes, scales)
PyObject* quant_rowwise_i8(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS AQ_ARGS(1);
  const Tensor* x = unpack(args[0]);
  Call c;
  Rows r;
  if (!x || !c.at(*x) || !rows_of(*x, &r)) return none();
  c.current_stream();
  Tensor q = c.empty({r.M, r.K}, ScalarType::Char), s = c.empty({r.M}, ScalarType::Float);
  const int rc = queued([&] {
    return lib.aq_quant_rowwise_i8(r.p, r.code, r.M, r.K, r.K, static_cast<int8_t*>(q.mutable_data_ptr()),
                                   static_cast<float*>(s.mutable_data_ptr()), c.stream);
  });
  return rc ? fail(rc, "aq_quant_rowwise_i8") : pair(q, s);
  END_HANDLE_TH_ERRORS
}

// rmsnorm_quant_rowwise_i8(x, gamma, eps) -> (codes, scales)
PyObject* rmsnorm_quant_rowwise_i8(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS AQ_ARGS(3);
  const Tensor *x = unpack(args[0]), *g = unpack(args[1]);
  Call c;
  Rows r;
  if (!x || !g || !c.at(*x) || !rows_of(*x, &r) || !plain(*g, x->scalar_type(), c.dev) || g->numel() != r.K) return none();
  const double eps = PyFloat_AsDouble(args[2]);
  if (eps == -1.0 && PyErr_Occurred()) return nullptr;
  c.current_stream();
  Tensor q = c.empty({r.M, r.K}, ScalarType::Char), s = c.empty({r.M}, ScalarType::Float);
  const int rc = queued([&] {
    return lib.aq_rmsnorm_quant_rowwise_i8(r.p, r.code, g->const_data_ptr(), r.code, static_cast<float>(eps), r.M, r.K, r.K,
                                           static_cast<int8_t*>(q.mutable_data_ptr()), static_cast<float*>(s.mutable_data_ptr()),
                                           c.stream);
  });
  return rc ? fail(rc, "aq_rmsnorm_quant_rowwise_i8") : pair(q, s);
  END_HANDLE_TH_ERRORS
}

// swiglu_quant_rowwise_i8(ug) -> (codes, scales)
PyObject* swiglu_quant_rowwise_i8(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS AQ_ARGS(1);
  const Tensor* x = unpack(args[0]);
  Call c;
  Rows r;
  if (!x || !c.at(*x) || !rows_of(*x, &r) || r.K % 32) return none();
  c.current_stream();
  const int64_t F = r.K / 2;
  Tensor q = c.empty({r.M, F}, ScalarType::Char), s = c.empty({r.M}, ScalarType::Float);
  const int rc = queued([&] {
    return lib.aq_swiglu_quant_rowwise_i8(r.p, r.code, r.M, F, r.K, static_cast<int8_t*>(q.mutable_data_ptr()),
                                          static_cast<float*>(s.mutable_data_ptr()), c.stream);
  });
  return rc ? fail(rc, "aq_swiglu_quant_rowwise_i8") : pair(q, s);
  END_HANDLE_TH_ERRORS
}

// gemv_w8a8_decode(x, wq, sw, bias, out_dtype, residual, gamma, eps) -> y [M, N]: at most 16 rows
PyObject* gemv_w8a8_decode(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS AQ_ARGS(8);
  const Tensor *x = unpack(args[0]), *w, *s;
  Call c;
  Rows r;
  Bias b;
  ScalarType type;
  const void* res;
  if (!x || !c.at(*x) || !rows_of(*x, &r) || r.M > 16 || !weight_of(args[1], args[2], r.K, c.dev, false, &w, &s)) return none();
  const int64_t N = w->size(0);
  if (!bias_of(args[3], N, c.dev, &b) || !out_type(args[4], x->scalar_type(), &type) ||
      !residual_of(args[5], r.M, N, type, c.dev, &res))
    return none();
  const Tensor* g = nullptr;
  double eps = 0.0;
  if (args[6] != Py_None) {
    g = unpack(args[6]);
    if (!g || !plain(*g, x->scalar_type(), c.dev) || g->numel() != r.K) return none();
    eps = PyFloat_AsDouble(args[7]);
    if (eps == -1.0 && PyErr_Occurred()) return nullptr;
  }
  c.current_stream();
  const size_t need = lib.aq_gemv_w8a8_workspace_bytes(r.M, r.K);
  Tensor y = c.empty({r.M, N}, type), ws = c.empty({static_cast<int64_t>(need)}, ScalarType::Byte);
  const auto* wp = static_cast<const int8_t*>(w->const_data_ptr());
  const auto* sp = static_cast<const float*>(s->const_data_ptr());
  const int rc = queued([&] {
    return g ? lib.aq_gemv_w8a8_decode_rmsnorm(r.p, r.code, g->const_data_ptr(), static_cast<float>(eps), wp, sp, b.p, b.code, res,
                                               y.mutable_data_ptr(), act_code(type), r.M, N, r.K, ws.mutable_data_ptr(), need,
                                               c.stream)
             : lib.aq_gemv_w8a8_decode_residual(r.p, r.code, wp, sp, b.p, b.code, res, y.mutable_data_ptr(), act_code(type), r.M,
                                                N, r.K, ws.mutable_data_ptr(), need, c.stream);
  });
  return rc ? fail(rc, "aq_gemv_w8a8_decode") : THPVariable_Wrap(y);
  END_HANDLE_TH_ERRORS
}

// (xq, sx, wq, sw, bias, out_dtype, residual) -> y [M, N] through one of the entry points that take codes
template <class Fn>
PyObject* on_codes(PyObject* const* args, bool fp8, int64_t max_rows, const char* what, Fn&& call) {
  const Tensor *xq = unpack(args[0]), *sx = unpack(args[1]), *w, *s;
  Call c;
  if (!xq || !sx || !c.at(*xq) || !plain(*xq, fp8 ? ScalarType::Byte : ScalarType::Char, c.dev) || xq->dim() != 2) return none();
  const int64_t M = xq->size(0), K = xq->size(1);
  if (M < 1 || M > max_rows || K < 16 || K % 16 || !aligned16(xq->const_data_ptr()) || !plain(*sx, ScalarType::Float, c.dev) ||
      sx->numel() != (fp8 ? 1 : M) || !weight_of(args[2], args[3], K, c.dev, fp8, &w, &s) || !THPDtype_Check(args[5]))
    return none();
  const int64_t N = w->size(0);
  const ScalarType type = reinterpret_cast<THPDtype*>(args[5])->scalar_type;
  Bias b;
  const void* res;
  if (act_code(type) < 0 || !bias_of(args[4], N, c.dev, &b) || !residual_of(args[6], M, N, type, c.dev, &res)) return none();
  c.current_stream();
  Tensor y = c.empty({M, N}, type);
  const int rc = queued([&] {
    return call(xq->const_data_ptr(), static_cast<const float*>(sx->const_data_ptr()), w->const_data_ptr(),
                static_cast<const float*>(s->const_data_ptr()), b, res, y.mutable_data_ptr(), act_code(type), M, N, K, c.stream);
  });
  return rc ? fail(rc, what) : THPVariable_Wrap(y);
}

#define AQ_ON_CODES(NAME, ENTRY, CODE, FP8, MAX_ROWS)                                                                       \
  PyObject* NAME(PyObject*, PyObject* const* args, Py_ssize_t nargs) {                                                      \
    HANDLE_TH_ERRORS AQ_ARGS(7);                                                                                            \
    return on_codes(args, FP8, MAX_ROWS, #ENTRY,                                                                            \
                    [](const void* xq, const float* sx, const void* w, const float* sw, const Bias& b, const void* res,     \
                       void* y, int y_code, int64_t M, int64_t N, int64_t K, void* stream) {                                \
                      return lib.ENTRY(static_cast<const CODE*>(xq), sx, static_cast<const CODE*>(w), sw, b.p, b.code, res, \
                                       y, y_code, M, N, K, stream);                                                         \
                    });                                                                                                     \
    END_HANDLE_TH_ERRORS                                                                                                    \
  }
AQ_ON_CODES(linear_w8a8, aq_linear_w8a8_residual, int8_t, false, INT64_MAX)
AQ_ON_CODES(gemv_w8a8_codes, aq_gemv_w8a8_codes_residual, int8_t, false, 16)
AQ_ON_CODES(linear_fp8, aq_linear_fp8_residual, uint8_t, true, INT64_MAX)

// gemv_fp8_decode(x, wq, sw, bias, out_dtype, residual) -> y [M, N]: at most 16 rows
PyObject* gemv_fp8_decode(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS AQ_ARGS(6);
  const Tensor *x = unpack(args[0]), *w, *s;
  Call c;
  Rows r;
  Bias b;
  ScalarType type;
  const void* res;
  if (!x || !c.at(*x) || !rows_of(*x, &r) || r.M > 16 || !weight_of(args[1], args[2], r.K, c.dev, true, &w, &s)) return none();
  const int64_t N = w->size(0);
  if (!bias_of(args[3], N, c.dev, &b) || !out_type(args[4], x->scalar_type(), &type) ||
      !residual_of(args[5], r.M, N, type, c.dev, &res))
    return none();
  c.current_stream();
  const size_t need = lib.aq_gemv_fp8_workspace_bytes(r.M, r.K);
  Tensor y = c.empty({r.M, N}, type), ws = c.empty({static_cast<int64_t>(need)}, ScalarType::Byte);
  const int rc = queued([&] {
    return lib.aq_gemv_fp8_decode_residual(r.p, r.code, static_cast<const uint8_t*>(w->const_data_ptr()),
                                           static_cast<const float*>(s->const_data_ptr()), b.p, b.code, res, y.mutable_data_ptr(),
                                           act_code(type), r.M, N, r.K, ws.mutable_data_ptr(), need, c.stream);
  });
  return rc ? fail(rc, "aq_gemv_fp8_decode") : THPVariable_Wrap(y);
  END_HANDLE_TH_ERRORS
}

// quant_tensor_fp8(x, state or None) -> (codes with x's shape, scale [1]); with the state: the one-launch form
PyObject* quant_tensor_fp8(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS AQ_ARGS(2);
  const Tensor* x = unpack(args[0]);
  Call c;
  if (!x || !c.at(*x) || act_code(x->scalar_type()) < 0 || !x->is_contiguous() || x->numel() % 16 || x->numel() == 0) return none();
  const Tensor* state = nullptr;
  if (args[1] != Py_None) {
    state = unpack(args[1]);
    if (!state || !plain(*state, ScalarType::Long, c.dev) || state->numel() * 8 < AQ_FP8_ONEPASS_WS_BYTES) return none();
  }
  c.current_stream();
  Tensor q = c.empty(x->sizes(), ScalarType::Byte), s = c.empty({1}, ScalarType::Float), ws;
  if (!state) ws = c.empty({AQ_FP8_AMAX_WS_BYTES}, ScalarType::Byte);
  const int rc = queued([&] {
    auto* qp = static_cast<uint8_t*>(q.mutable_data_ptr());
    auto* sp = static_cast<float*>(s.mutable_data_ptr());
    return state ? lib.aq_quant_tensor_fp8_onepass(x->const_data_ptr(), act_code(x->scalar_type()), x->numel(), qp, sp,
                                                   state->mutable_data_ptr(), state->numel() * 8, c.stream)
                 : lib.aq_quant_tensor_fp8(x->const_data_ptr(), act_code(x->scalar_type()), x->numel(), qp, sp,
                                           static_cast<uint32_t*>(ws.mutable_data_ptr()), AQ_FP8_AMAX_WS_BYTES, c.stream);
  });
  return rc ? fail(rc, state ? "aq_quant_tensor_fp8_onepass" : "aq_quant_tensor_fp8") : pair(q, s);
  END_HANDLE_TH_ERRORS
}

// ---- module attributes, read where nn.Module keeps them ----------------------------------------------------------
// nn.Module.__getattr__ costs about half a microsecond a name; a fused block names thirty.

PyObject *k_modules, *k_buffers, *k_parameters, *k_qweight, *k_w_scale, *k_bias, *k_weight, *k_norm_eps, *k_forward, *k_fwd_hooks,
    *k_fwd_pre_hooks, *k_compiled, *k_attention, *k_mlp, *k_input_norm, *k_post_norm, *k_qkv, *k_upgate, *k_o_proj, *k_down, *k_q_norm,
    *k_k_norm, *k_decode_attention, *k_use_qk_norm, *k_use_gate, *k_n_heads, *k_n_kv_heads, *k_head_dim, *k_layer_id, *k_swiglu_quant,
    *k_norm_quant, *k_residual_adds, *k_k_layers, *k_v_layers, *k_page_table, *k_total_len, *k_seq_lens, *k_invalid, *k_page_size,
    *k_shared, *k_residual, *k_norm, *k_call, *k_decode_rows, *k_forward_codes, *k_forward_attn;

PyObject* dict_of(PyObject* o) {  // borrowed; null if it has none
  PyObject** d = _PyObject_GetDictPtr(o);
  return d && *d && PyDict_Check(*d) ? *d : nullptr;
}
PyObject* get(PyObject* d, PyObject* key) {  // borrowed
  return d && PyDict_Check(d) ? PyDict_GetItem(d, key) : nullptr;
}
PyObject* nested(PyObject* d, PyObject* group, PyObject* key) { return get(get(d, group), key); }
bool truth(PyObject* d, PyObject* key) { return get(d, key) == Py_True; }
bool integer(PyObject* d, PyObject* key, int64_t* v) {
  PyObject* o = get(d, key);
  if (!o || !PyLong_CheckExact(o)) return false;
  *v = PyLong_AsLongLong(o);
  return true;
}

// A class, and what its instances' calls go through as the package defined it: (class, name, value) for each method.
struct Class {
  PyObject *type = nullptr, *defined = nullptr;
  unsigned version = 0;  // the class's tag when it last was as defined
};

// No method has been replaced, on the class, one of its bases or nn.Module.  A class that changes, or one of whose bases
// does, loses its version tag, which is never used twice: usually one compare.
bool as_defined(Class& c) {
#if PY_VERSION_HEX < 0x030c0000
  const auto* t = reinterpret_cast<PyTypeObject*>(c.type);
  const bool tagged = PyType_HasFeature(const_cast<PyTypeObject*>(t), Py_TPFLAGS_VALID_VERSION_TAG);
  if (tagged && c.version && c.version == t->tp_version_tag) return true;
#endif
  for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(c.defined); ++i) {
    PyObject* d = PyTuple_GET_ITEM(c.defined, i);
    if (_PyType_Lookup(reinterpret_cast<PyTypeObject*>(PyTuple_GET_ITEM(d, 0)), PyTuple_GET_ITEM(d, 1)) != PyTuple_GET_ITEM(d, 2)) return false;
  }
#if PY_VERSION_HEX < 0x030c0000
  c.version = PyType_HasFeature(const_cast<PyTypeObject*>(t), Py_TPFLAGS_VALID_VERSION_TAG) ? t->tp_version_tag : 0;
#endif
  return true;
}

// {class: ((class, name, value), ...)} as linear.as_defined() makes it; held for the life of the process
bool take_class(PyObject* classes, PyObject* type, Class* c) {
  PyObject* defined = PyDict_GetItem(classes, type);
  if (!PyType_Check(type) || !defined || !PyTuple_CheckExact(defined)) return false;
  for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(defined); ++i) {
    PyObject* d = PyTuple_GET_ITEM(defined, i);
    if (!PyTuple_CheckExact(d) || PyTuple_GET_SIZE(d) != 3 || !PyType_Check(PyTuple_GET_ITEM(d, 0)) || !PyUnicode_CheckExact(PyTuple_GET_ITEM(d, 1)))
      return false;
  }
  Py_INCREF(type);
  Py_INCREF(defined);
  *c = {type, defined, 0};
  return true;
}

// What the functions that stand for a module's call are told about the Python side, once (set_linear_types, set_block_types).
struct Types {
  Class quant_linear, fp8_linear, gqa, mlp, paged_kv;
  PyObject* global_hooks = nullptr;  // tuple of the dicts of hooks that run for every module
  PyObject* ops_dict = nullptr;      // the operators' module and, by name, the operators as they were defined
  PyObject *linear_ops = nullptr, *block_ops = nullptr;
  uint64_t linear_ops_version = 0, block_ops_version = 0;  // of ops_dict when it last held them all
  PyObject *rms_norm = nullptr, *native_call = nullptr;
  // Limits, as the Python side had them when it was imported.  A call goes the general way while one of them is another.
  int64_t decode_rows = 0, fp8_decode_rows = 0, fp8_onepass_min_bytes = 0;
  struct Merge {
    int64_t rows, width, slices, slice, work;
  } merge = {};
  PyObject *norm_max_k = nullptr, *swiglu_max_f = nullptr;  // {dtype: limit}, read at each call
} types;

// whole numbers, all positive, from a tuple
bool limits_of(PyObject* t, std::initializer_list<int64_t*> to) {
  if (!PyTuple_Check(t) || PyTuple_GET_SIZE(t) != static_cast<Py_ssize_t>(to.size())) return false;
  Py_ssize_t i = 0;
  for (int64_t* v : to) {
    PyObject* o = PyTuple_GET_ITEM(t, i++);
    if (!PyLong_CheckExact(o) || (*v = PyLong_AsLongLong(o)) < 1) return false;
  }
  return true;
}

bool exactly(PyObject* o, PyObject* type) { return o && reinterpret_cast<PyObject*>(Py_TYPE(o)) == type; }

// A module whose forward may be replaced by what it is known to do: exactly the class, as it was defined, nothing hooked,
// nothing wrapped, no row limit of its own.
bool ordinary(PyObject* m, Class& c) {
  if (!exactly(m, c.type) || !as_defined(c)) return false;
  PyObject* d = dict_of(m);
  if (!d || PyDict_GetItem(d, k_forward) || PyDict_GetItem(d, k_decode_rows)) return false;
  PyObject *h = get(d, k_fwd_hooks), *p = get(d, k_fwd_pre_hooks), *comp = get(d, k_compiled);
  return (!h || (PyDict_Check(h) && PyDict_GET_SIZE(h) == 0)) && (!p || (PyDict_Check(p) && PyDict_GET_SIZE(p) == 0)) &&
         (!comp || comp == Py_None);
}

// Nothing watches module calls globally, and the operators are the package's own: a program that replaces one (to
// count or trace calls) has every call go through its replacement, on the step-by-step path.
// The operators' dictionary is looked through again only once it has changed (its version tag is never used twice).
bool unobserved(PyObject* operators) {
  for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(types.global_hooks); ++i)
    if (PyDict_GET_SIZE(PyTuple_GET_ITEM(types.global_hooks, i))) return false;
#if PY_VERSION_HEX < 0x030c0000
  uint64_t& seen = operators == types.block_ops ? types.block_ops_version : types.linear_ops_version;
  const uint64_t version = reinterpret_cast<PyDictObject*>(types.ops_dict)->ma_version_tag;
  if (seen == version) return true;
#endif
  PyObject *name, *own;
  Py_ssize_t at = 0;
  while (PyDict_Next(operators, &at, &name, &own))
    if (PyDict_GetItem(types.ops_dict, name) != own) return false;
#if PY_VERSION_HEX < 0x030c0000
  seen = version;
#endif
  return true;
}

struct Proj {  // a QuantLinear's tensors, held for the length of the call
  Tensor hold_w, hold_s;
  const int8_t* w = nullptr;
  const float* s = nullptr;
  Bias b;
  int64_t N = 0, K = 0;
};
bool proj_of(PyObject* m, int dev, Proj* p) {
  if (!ordinary(m, types.quant_linear)) return false;
  PyObject* d = dict_of(m);
  if (get(d, k_shared) != Py_None) return false;
  const Tensor *w = unpack(nested(d, k_buffers, k_qweight)), *s = unpack(nested(d, k_buffers, k_w_scale));
  if (!w || !s || w->dim() != 2 || !plain(*w, ScalarType::Char, dev) || !plain(*s, ScalarType::Float, dev)) return false;
  p->N = w->size(0);
  p->K = w->size(1);
  if (s->numel() != p->N || p->K % 16 || !aligned16(w->const_data_ptr())) return false;
  PyObject* bias = nested(d, k_parameters, k_bias);
  if (!bias_of(bias ? bias : get(d, k_bias), p->N, dev, &p->b)) return false;
  p->hold_w = *w;
  p->hold_s = *s;
  p->w = static_cast<const int8_t*>(w->const_data_ptr());
  p->s = static_cast<const float*>(s->const_data_ptr());
  return true;
}

struct Gain {
  Tensor hold;
  const void* p = nullptr;
  float eps = 0.f;
};
bool gain_of(PyObject* m, int64_t K, int dev, Gain* g) {
  if (!exactly(m, types.rms_norm)) return false;  // not called: its tensors are read
  PyObject* d = dict_of(m);
  const Tensor* w = unpack(nested(d, k_parameters, k_weight));
  PyObject* eps = get(d, k_norm_eps);
  if (!w || !plain(*w, ScalarType::BFloat16, dev) || w->numel() != K || !aligned16(w->const_data_ptr()) || !eps ||
      !PyFloat_CheckExact(eps) || !(PyFloat_AS_DOUBLE(eps) >= 0.0))
    return false;
  g->hold = *w;
  g->p = w->const_data_ptr();
  g->eps = static_cast<float>(PyFloat_AS_DOUBLE(eps));
  return true;
}

// What calling the QuantLinear or Fp8Linear gives, or None where nn.Module's own call has to serve: hooks, a shared input, FP8
// inputs that are quantised in one launch with a state the module keeps.
PyObject* linear_native(PyObject* layer, PyObject* const* args, Py_ssize_t nargs, PyObject* names) {
  HANDLE_TH_ERRORS
  const bool fp8 = exactly(layer, types.fp8_linear.type);
  if (!lib.aq_error_string || !types.linear_ops || nargs != 1 || !ordinary(layer, fp8 ? types.fp8_linear : types.quant_linear) ||
      !unobserved(types.linear_ops))
    return none();
  PyObject *residual = nullptr, *norm = nullptr;
  for (Py_ssize_t i = 0; names && i < PyTuple_GET_SIZE(names); ++i) {
    PyObject* name = PyTuple_GET_ITEM(names, i);  // interned, as keyword names are; another text of the same value takes the general path
    if (name == k_residual)
      residual = args[1 + i];
    else if (name == k_norm && !fp8)
      norm = args[1 + i] == Py_None ? nullptr : args[1 + i];
    else
      return none();
  }
  PyObject* d = dict_of(layer);
  if (!fp8 && get(d, k_shared) != Py_None) return none();
  const Tensor *x = unpack(args[0]), *w, *s;
  Call c;
  Rows r;
  Bias b;
  const void* res;
  PyObject *wq = nested(d, k_buffers, k_qweight), *sw = nested(d, k_buffers, k_w_scale);
  if (!x || x->requires_grad() || !c.at(*x) || !rows_of(*x, &r) || !weight_of(wq, sw, r.K, c.dev, fp8, &w, &s)) return none();
  const Held hold_w(wq), hold_s(sw);  // the module may be given others while the interpreter lock is released
  const int64_t N = w->size(0);
  const ScalarType type = x->scalar_type();
  PyObject* bias = nested(d, k_parameters, k_bias);
  if (!bias_of(bias ? bias : get(d, k_bias), N, c.dev, &b) || !residual_of(residual, r.M, N, type, c.dev, &res)) return none();
  const void* gain = nullptr;
  float eps = 0.f;
  if (norm) {
    if (!PyTuple_CheckExact(norm) || PyTuple_GET_SIZE(norm) != 2 || !PyFloat_CheckExact(PyTuple_GET_ITEM(norm, 1))) return none();
    const Tensor* g = unpack(PyTuple_GET_ITEM(norm, 0));
    if (!g || !plain(*g, type, c.dev) || g->numel() != r.K) return none();
    gain = g->const_data_ptr();
    eps = static_cast<float>(PyFloat_AS_DOUBLE(PyTuple_GET_ITEM(norm, 1)));
  }
  const int64_t x_bytes = x->numel() * x->element_size();
  const bool few = r.M <= (fp8 ? types.fp8_decode_rows : types.decode_rows);
  if (fp8 && !few && x_bytes >= types.fp8_onepass_min_bytes) return none();
  c.current_stream();
  c10::DimVector shape(x->sizes());
  shape.back() = N;
  Tensor y = c.empty(shape, type);
  // codes and scales of the tokens (and, for FP8, the partial maxima); the codes of a tile's rows begin on lines
  const int64_t pitch = few || gain ? r.K : lib.aq_linear_codes_pitch(fp8, res != nullptr, r.M, N, r.K);
  const int64_t codes = !few  ? (r.M * pitch + 255) & ~int64_t(255)
                        : fp8 ? static_cast<int64_t>(lib.aq_gemv_fp8_workspace_bytes(r.M, r.K))
                              : static_cast<int64_t>(lib.aq_gemv_w8a8_workspace_bytes(r.M, r.K));
  const int64_t room = codes + (!few ? (fp8 ? 256 + AQ_FP8_AMAX_WS_BYTES : 4 * r.M) : 0);
  void* yp = y.mutable_data_ptr();
  // a launch that quantises its rows itself touches no workspace: an allocation is 0.4 us of a 5 us call
  const bool tiles = !few && lib.aq_linear_few_rows_ok(r.code, gain != nullptr, fp8, r.M, N, r.K) &&
                     (!c.captured() || lib.aq_linear_few_rows_queued_ok(r.code, gain != nullptr, fp8, r.M, N, r.K));
  const bool alone = tiles || (few && (fp8 ? lib.aq_gemv_fp8_decode_one_launch(r.code, r.M, r.K)
                                 : lib.aq_gemv_w8a8_decode_one_launch(r.code, gain != nullptr, r.M, N, r.K)));
  Tensor ws;
  if (!alone) ws = c.empty({room}, ScalarType::Byte);
  char* base = static_cast<char*>(alone ? yp : ws.mutable_data_ptr());
  auto* sx = reinterpret_cast<float*>(base + codes);
  const void* wp = w->const_data_ptr();
  const auto* sp = static_cast<const float*>(s->const_data_ptr());
  const char* what = "";
  const int rc = queued([&]() -> int {
    if (tiles) {
      what = "aq_linear_few_rows";
      return lib.aq_linear_few_rows(r.p, r.code, gain, eps, wp, fp8, sp, b.p, b.code, res, yp, r.code, r.M, N, r.K, c.stream);
    }
    if (few) {
      what = fp8 ? "aq_gemv_fp8_decode" : "aq_gemv_w8a8_decode";
      if (fp8)
        return lib.aq_gemv_fp8_decode_residual(r.p, r.code, static_cast<const uint8_t*>(wp), sp, b.p, b.code, res, yp, r.code, r.M, N, r.K,
                                               base, codes, c.stream);
      if (gain)
        return lib.aq_gemv_w8a8_decode_rmsnorm(r.p, r.code, gain, eps, static_cast<const int8_t*>(wp), sp, b.p, b.code, res, yp, r.code,
                                               r.M, N, r.K, base, codes, c.stream);
      return lib.aq_gemv_w8a8_decode_residual(r.p, r.code, static_cast<const int8_t*>(wp), sp, b.p, b.code, res, yp, r.code, r.M, N, r.K,
                                              base, codes, c.stream);
    }
    if (fp8) {
      auto* q = reinterpret_cast<uint8_t*>(base);
      what = "aq_quant_tensor_fp8";
      auto* maxima = reinterpret_cast<uint32_t*>(base + codes + 256);
      if (int e = pitch != r.K ? lib.aq_quant_tensor_fp8_strided(r.p, r.code, r.M, r.K, q, pitch, sx, maxima, AQ_FP8_AMAX_WS_BYTES, c.stream)
                               : lib.aq_quant_tensor_fp8(r.p, r.code, x->numel(), q, sx, maxima, AQ_FP8_AMAX_WS_BYTES, c.stream))
        return e;
      what = "aq_linear_fp8";
      if (pitch != r.K)
        return lib.aq_linear_fp8_strided(q, pitch, sx, static_cast<const uint8_t*>(wp), sp, b.p, b.code, res, yp, r.code, r.M, N, r.K, c.stream);
      return lib.aq_linear_fp8_residual(q, sx, static_cast<const uint8_t*>(wp), sp, b.p, b.code, res, yp, r.code, r.M, N, r.K, c.stream);
    }
    auto* q = reinterpret_cast<int8_t*>(base);
    what = gain ? "aq_rmsnorm_quant_rowwise_i8" : "aq_quant_rowwise_i8";
    if (int e = gain           ? lib.aq_rmsnorm_quant_rowwise_i8(r.p, r.code, gain, r.code, eps, r.M, r.K, r.K, q, sx, c.stream)
                : pitch != r.K ? lib.aq_quant_rowwise_i8_strided(r.p, r.code, r.M, r.K, r.K, q, pitch, sx, c.stream)
                               : lib.aq_quant_rowwise_i8(r.p, r.code, r.M, r.K, r.K, q, sx, c.stream))
      return e;
    what = "aq_linear_w8a8";
    if (pitch != r.K)
      return lib.aq_linear_w8a8_strided(q, pitch, sx, static_cast<const int8_t*>(wp), sp, b.p, b.code, res, yp, r.code, r.M, N, r.K, c.stream);
    return lib.aq_linear_w8a8_residual(q, sx, static_cast<const int8_t*>(wp), sp, b.p, b.code, res, yp, r.code, r.M, N, r.K, c.stream);
  });
  return rc ? fail(rc, what) : THPVariable_Wrap(y);
  END_HANDLE_TH_ERRORS
}

// The call of the quantized layers' __call__, a Python function of _NativeCall: its own code is what a compiler that traces
// the call reads (a method written in C it could not).  What linear_native does not take goes where that code would send
// it, the next __call__ behind _NativeCall, nn.Module's as a rule; a subclass or a module with hooks is 0.5 us faster so.
PyObject* linear_call(PyObject* function, PyObject* const* args, size_t nargsf, PyObject* names) {
  const Py_ssize_t nargs = PyVectorcall_NARGS(nargsf);
  if (nargs > 0) {
    PyObject* y = linear_native(args[0], args + 1, nargs - 1, names);
    if (y != Py_None) return y;
    Py_DECREF(y);
    PyObject* mro = Py_TYPE(args[0])->tp_mro;
    bool behind = false;
    for (Py_ssize_t i = 0; mro && i < PyTuple_GET_SIZE(mro); ++i) {
      PyObject* c = PyTuple_GET_ITEM(mro, i);
      PyObject* next = behind ? get(reinterpret_cast<PyTypeObject*>(c)->tp_dict, k_call) : nullptr;
      if (next && !PyFunction_Check(next)) break;  // something that binds in its own way
      if (next) {
        const Held held(next);
        return PyObject_Vectorcall(next, args, nargsf, names);
      }
      behind = behind || c == types.native_call;
    }
  }
  return _PyFunction_Vectorcall(function, args, nargsf, names);
}

// serve_calls(_NativeCall): has calls of its __call__ come to linear_call
PyObject* serve_calls(PyObject*, PyObject* cls) {
  PyObject* function = PyType_Check(cls) ? get(reinterpret_cast<PyTypeObject*>(cls)->tp_dict, k_call) : nullptr;
  if (!function || !PyFunction_Check(function)) return PyErr_Format(PyExc_TypeError, "serve_calls");
  Py_INCREF(cls);  // for the life of the process
  types.native_call = cls;
#if PY_VERSION_HEX >= 0x030c0000
  PyFunction_SetVectorcall(reinterpret_cast<PyFunctionObject*>(function), linear_call);
#else
  reinterpret_cast<PyFunctionObject*>(function)->vectorcall = linear_call;
#endif
  Py_RETURN_NONE;
}

// set_linear_types(QuantLinear, Fp8Linear, {class: what it defines}, hook dicts, ops.__dict__, {name: operator or limit as defined},
//                  (row limit, row limit, bytes from which FP8 inputs are quantised in one launch))
PyObject* set_linear_types(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  AQ_ARGS(7);
  if (!PyDict_Check(args[2]) || !take_class(args[2], args[0], &types.quant_linear) || !take_class(args[2], args[1], &types.fp8_linear) ||
      !PyTuple_Check(args[3]) || !PyDict_Check(args[4]) || !PyDict_Check(args[5]) ||
      !limits_of(args[6], {&types.decode_rows, &types.fp8_decode_rows, &types.fp8_onepass_min_bytes}))
    return PyErr_Format(PyExc_TypeError, "set_linear_types");
  for (Py_ssize_t i = 3; i < 6; ++i) Py_INCREF(args[i]);  // for the life of the process
  types.global_hooks = args[3], types.ops_dict = args[4], types.linear_ops = args[5];
  Py_RETURN_NONE;
}

// One stretch of device memory that a block's intermediate results are cut from.
struct Scratch {
  char* base = nullptr;
  size_t used = 0, most = 0;
  size_t take(size_t bytes) {
    const size_t at = used;
    used += (bytes + 255) & ~static_cast<size_t>(255);
    if (used > most) most = used;
    return at;
  }
};

// ops.attn_gemv_fusable: whether the output projection merges the attention's slices itself
bool merge_in_projection(int64_t B, int64_t width, int64_t total) {
  const Types::Merge& m = types.merge;
  if (B < 1 || B > m.rows || width > m.width || total <= m.slice || total > m.slices * m.slice) return false;
  return B * width * ((total + m.slice - 1) / m.slice) <= m.work;
}

// attn_gemv_fusable(B, width, total) -> bool, for comparison with the operator's rule
PyObject* attn_gemv_fusable(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  AQ_ARGS(3);
  int64_t v[3];
  for (int i = 0; i < 3; ++i)
    if ((v[i] = PyLong_AsLongLong(args[i])) == -1 && PyErr_Occurred()) return nullptr;
  return PyBool_FromLong(types.block_ops && merge_in_projection(v[0], v[1], v[2]));
}

// an operator's limit for bf16 rows: its entry in {dtype: limit}
int64_t limit_of(PyObject* by_type) {
  PyObject* v = get(by_type, reinterpret_cast<PyObject*>(torch::getTHPDtype(ScalarType::BFloat16)));
  return v && PyLong_CheckExact(v) ? PyLong_AsLongLong(v) : 0;
}

// A DecoderBlock with every fusion on (fuse_shared_inputs(norms, decode_attention, residuals)), applied to bf16 tokens over
// a paged cache: what it works on, read and checked under the interpreter lock.
struct Block {
  Call c;
  int64_t B, S, M, dim, Hq, Hkv, D, F, total, P, page, n_pages, fr_stride, swiglu_gemv;
  const float* fr;
  const int64_t* table;
  const int64_t* lens = nullptr;
  char *kc, *vc;
  bool direct, qk_norm;
  float scale;
  Tensor hold_x, hold_fr, hold_k, hold_v, hold_table, hold_lens;
  Proj qkv, o, ug, down;
  Gain n1, n2, qn, kn;

  // the intermediate results' places in the scratch memory, `most` bytes
  size_t x1, sx, qkv_rows, att, codes, q, k, parts, up_gate, h_codes, most;
  int64_t parts_bytes;

  bool read(PyObject* block, PyObject* x, PyObject* rotary, PyObject* cache);
  void lay_out();
  bool few() const { return M <= types.decode_rows; }
  bool step() const { return S == 1; }
  // Whether a prompt's attention rotates its queries itself, which then are not written and read back: from 4 MB of them on, 8 MB with
  // qk-norm.  With less, the launch that rotates takes the same few microseconds whatever it moves, and rotating (qk-norm: and a sum
  // over the head) is one more link in the attention launch's chain.  us a block, rotated before -> in attention:
  //   16 heads of 128, MB of queries: 1.0 64.1 -> 64.6, 2.8 96.7 -> 97.3, 3.1 104.4 -> 104.1, 4.2 108.5 -> 108.4, 4.6 124.2 -> 123.6,
  //     5.9 137.0 -> 136.2, 8.4 156.9 -> 154.6, 16.4 268.1 -> 264.6; with qk-norm 3.9 104.8 -> 106.6, 5.6 139.7 -> 141.3, 7.9 160.1 ->
  //     161.1, 8.4 157.1 -> 156.5, 10.5 189.7 -> 189.0, 16.8 271.8 -> 268.2;
  //   24 heads of 64: 0.8 58.4 -> 59.1, 2.1 83.8 -> 83.6, 2.9 108.6 -> 109.1, 3.9 116.2 -> 115.6, 4.7 125.3 -> 124.7, 6.3 143.5 -> 142.3, 8.4 186.4
  //     -> 184.3; with qk-norm 3.1 99.8 -> 101.1, 6.3 146.3 -> 146.6, 7.9 168.5 -> 167.6, 11.8 222.0 -> 219.4.
  // (48 + 52 sizes, on an empty cache and on top of tokens; on this side of the line 0.2 to 1.5 % faster, one in ten level or 0.4 % slower.)
  bool rotates() const { return !step() && M * Hq * D >= (int64_t(qk_norm ? 4 : 2) << 20); }
  bool merge() const { return step() && merge_in_projection(B, Hq * D, total); }
  int queue(const void* in, void* out, char* base, const char** what) const;  // allocates nothing: runs without the interpreter lock
};

bool Block::read(PyObject* block, PyObject* px, PyObject* protary, PyObject* cache) {
  // the tokens
  const Tensor *x = unpack(px), *rot = unpack(protary);
  if (!x || !rot || !c.at(*x) || !plain(*x, ScalarType::BFloat16, c.dev) || x->dim() != 3) return false;
  B = x->size(0), S = x->size(1), dim = x->size(2), M = B * S;
  if (M < 1 || dim > limit_of(types.norm_max_k) || !aligned16(x->const_data_ptr()) || x->requires_grad()) return false;
  hold_x = *x;
  // the modules
  PyObject* d = dict_of(block);
  if (!d || !truth(d, k_norm_quant) || !truth(d, k_residual_adds)) return false;
  PyObject *att = nested(d, k_modules, k_attention), *mlp = nested(d, k_modules, k_mlp);
  if (!ordinary(att, types.gqa) || !ordinary(mlp, types.mlp)) return false;
  PyObject *ad = dict_of(att), *md = dict_of(mlp);
  int64_t layer;
  if (!truth(ad, k_decode_attention) || !truth(md, k_swiglu_quant) || get(ad, k_use_gate) != Py_False || !integer(ad, k_n_heads, &Hq) ||
      !integer(ad, k_n_kv_heads, &Hkv) || !integer(ad, k_head_dim, &D) || !integer(ad, k_layer_id, &layer))
    return false;
  qk_norm = truth(ad, k_use_qk_norm);
  PyObject *po = nested(ad, k_modules, k_o_proj), *pdown = nested(md, k_modules, k_down);
  if (!proj_of(get(ad, k_qkv), c.dev, &qkv) || !proj_of(po, c.dev, &o) || get(dict_of(po), k_forward_attn) ||
      !proj_of(get(md, k_upgate), c.dev, &ug) || !proj_of(pdown, c.dev, &down) || get(dict_of(pdown), k_forward_codes) ||
      !gain_of(nested(d, k_modules, k_input_norm), dim, c.dev, &n1) || !gain_of(nested(d, k_modules, k_post_norm), dim, c.dev, &n2))
    return false;
  if (qk_norm && (!gain_of(nested(ad, k_modules, k_q_norm), D, c.dev, &qn) || !gain_of(nested(ad, k_modules, k_k_norm), D, c.dev, &kn)))
    return false;
  F = ug.N / 2;
  if (qkv.K != dim || qkv.N != (Hq + 2 * Hkv) * D || o.K != Hq * D || o.N != dim || ug.K != dim || ug.N % 2 || F % 16 ||
      F > limit_of(types.swiglu_max_f) || down.K != F || down.N != dim)
    return false;
  // the cache
  if (!exactly(cache, types.paged_kv.type) || !as_defined(types.paged_kv)) return false;
  PyObject* cd = dict_of(cache);
  const Tensor *k = unpack(get(cd, k_k_layers)), *v = unpack(get(cd, k_v_layers)), *t = unpack(get(cd, k_page_table));
  if (!k || !v || !t || !integer(cd, k_total_len, &total) || !integer(cd, k_page_size, &page)) return false;
  if (k->dim() != 5 || k->sizes() != v->sizes() || !plain(*k, ScalarType::BFloat16, c.dev) || !plain(*v, ScalarType::BFloat16, c.dev) ||
      layer < 0 || layer >= k->size(0) || k->size(2) != page || k->size(3) != Hkv || k->size(4) != D)
    return false;
  n_pages = k->size(1);
  if (!plain(*t, ScalarType::Long, c.dev) || t->dim() != 2 || t->size(0) != B) return false;
  P = t->size(1);
  if (total < S || total > P * page) return false;
  const int64_t layer_bytes = 2 * n_pages * page * Hkv * D;
  kc = static_cast<char*>(k->mutable_data_ptr()) + layer * layer_bytes;
  vc = static_cast<char*>(v->mutable_data_ptr()) + layer * layer_bytes;
  table = static_cast<const int64_t*>(t->const_data_ptr());
  hold_k = *k, hold_v = *v, hold_table = *t;
  PyObject* sl = get(cd, k_seq_lens);
  if (sl != Py_None) {
    const Tensor* l = unpack(sl);
    if (!l || !plain(*l, ScalarType::Long, c.dev) || l->dim() != 1 || l->size(0) != B) return false;
    lens = static_cast<const int64_t*>(l->const_data_ptr());
    hold_lens = *l;
  }
  direct = total == S && get(cd, k_invalid) == Py_None;
  // the rotary table: complex64 [B, S, D / 2], one stretch per sequence or one for all
  if (rot->scalar_type() != ScalarType::ComplexFloat || !rot->is_cuda() || rot->get_device() != c.dev || rot->is_conj() || rot->dim() != 3 ||
      rot->size(0) != B || rot->size(1) != S || rot->size(2) != D / 2 || rot->stride(2) != 1 || (S > 1 && rot->stride(1) != D / 2))
    return false;
  if (B == 1)
    fr_stride = S * D;
  else if (rot->stride(0) == 0 || rot->stride(0) == S * (D / 2))
    fr_stride = 2 * rot->stride(0);
  else
    return false;
  fr = static_cast<const float*>(rot->const_data_ptr());
  hold_fr = *rot;
  if (!aligned16(fr)) return false;
  scale = static_cast<float>(1.0 / std::sqrt(static_cast<double>(D)));
  swiglu_gemv = lib.aq_gemv_w8a8_decode_swiglu_ok(AQ_BF16, M, F, dim);
  c.current_stream();
  return true;
}

void Block::lay_out() {
  const int64_t A = Hq * D, KV = Hkv * D, longest = dim > A ? dim : A, widest = F > dim ? F : dim;
  Scratch m;
  x1 = m.take(2 * M * dim), sx = m.take(4 * M);
  const size_t shared = m.used;
  // attention
  qkv_rows = m.take(2 * M * qkv.N), att = m.take(2 * M * A);
  codes = m.take(few() ? lib.aq_gemv_w8a8_workspace_bytes(M, longest) : static_cast<size_t>(M * longest));
  q = step() || rotates() ? 0 : m.take(2 * M * A), k = step() || !direct ? 0 : m.take(2 * M * KV);
  parts_bytes = !step()   ? 0
                : merge() ? lib.aq_paged_attn_decode_partials_bytes(B, Hq, total)
                          : lib.aq_paged_attn_decode_workspace_bytes(B, Hq, Hkv, total);
  parts = m.take(static_cast<size_t>(parts_bytes));
  // the MLP, over the attention's results
  m.used = shared;
  up_gate = m.take(2 * M * (swiglu_gemv ? F : 2 * F));
  h_codes = m.take(few() ? lib.aq_gemv_w8a8_workspace_bytes(M, widest) : static_cast<size_t>(M * widest));
  most = m.most;
}

// Queues the block's launches: the ones, in the order and with the operands, of the step-by-step path in block.py, but that a prompt's
// queries may be rotated in its attention instead of before it (rotates()), and a small prompt's rows quantised in the launch that
// multiplies them (aq_linear_few_rows); the same bits.
int Block::queue(const void* in, void* out, char* base, const char** what) const {
  const bool few = this->few();
  const int64_t W = qkv.N, A = Hq * D, KV = Hkv * D;
  void* x1 = base + this->x1;
  float* sx = reinterpret_cast<float*>(base + this->sx);

  // y = projection of normalised tokens / of tokens as they are (+ residual); codes: room for M rows of the projection's K
  auto normed = [&](const Proj& p, const Gain& g, const void* x, void* y, size_t at) {
    void* room = base + at;
    if (few) {
      *what = "aq_gemv_w8a8_decode_rmsnorm";
      return lib.aq_gemv_w8a8_decode_rmsnorm(x, AQ_BF16, g.p, g.eps, p.w, p.s, p.b.p, p.b.code, nullptr, y, AQ_BF16, M, p.N, p.K, room,
                                             lib.aq_gemv_w8a8_workspace_bytes(M, p.K), c.stream);
    }
    if (lib.aq_linear_few_rows_queued_ok(AQ_BF16, 1, 0, M, p.N, p.K)) {
      *what = "aq_linear_few_rows";
      return lib.aq_linear_few_rows(x, AQ_BF16, g.p, g.eps, p.w, 0, p.s, p.b.p, p.b.code, nullptr, y, AQ_BF16, M, p.N, p.K, c.stream);
    }
    *what = "aq_rmsnorm_quant_rowwise_i8";
    int rc = lib.aq_rmsnorm_quant_rowwise_i8(x, AQ_BF16, g.p, AQ_BF16, g.eps, M, p.K, p.K, static_cast<int8_t*>(room), sx, c.stream);
    if (rc) return rc;
    *what = "aq_linear_w8a8";
    return lib.aq_linear_w8a8_residual(static_cast<const int8_t*>(room), sx, p.w, p.s, p.b.p, p.b.code, nullptr, y, AQ_BF16, M, p.N, p.K,
                                       c.stream);
  };
  auto projected = [&](const Proj& p, const void* x, const void* res, void* y, size_t at) {
    void* room = base + at;
    if (few) {
      *what = "aq_gemv_w8a8_decode";
      return lib.aq_gemv_w8a8_decode_residual(x, AQ_BF16, p.w, p.s, p.b.p, p.b.code, res, y, AQ_BF16, M, p.N, p.K, room,
                                              lib.aq_gemv_w8a8_workspace_bytes(M, p.K), c.stream);
    }
    if (lib.aq_linear_few_rows_queued_ok(AQ_BF16, 0, 0, M, p.N, p.K)) {
      *what = "aq_linear_few_rows";
      return lib.aq_linear_few_rows(x, AQ_BF16, nullptr, 0.f, p.w, 0, p.s, p.b.p, p.b.code, res, y, AQ_BF16, M, p.N, p.K, c.stream);
    }
    *what = "aq_quant_rowwise_i8";
    int rc = lib.aq_quant_rowwise_i8(x, AQ_BF16, M, p.K, p.K, static_cast<int8_t*>(room), sx, c.stream);
    if (rc) return rc;
    *what = "aq_linear_w8a8";
    return lib.aq_linear_w8a8_residual(static_cast<const int8_t*>(room), sx, p.w, p.s, p.b.p, p.b.code, res, y, AQ_BF16, M, p.N, p.K,
                                       c.stream);
  };

  char *q = base + qkv_rows, *att = base + this->att, *parts = base + this->parts;
  int rc = normed(qkv, n1, in, q, codes);
  if (rc) return rc;
  if (step()) {
    *what = "aq_rope_paged_attn_decode";
    if (merge()) {
      rc = qk_norm ? lib.aq_rope_paged_attn_decode_partials_qknorm(q, fr, fr_stride, table, P, total, lens, page, kc, vc, n_pages, scale, B,
                                                                   Hq, Hkv, D, qn.p, kn.p, qn.eps, parts, parts_bytes, c.stream)
                   : lib.aq_rope_paged_attn_decode_partials(q, fr, fr_stride, table, P, total, lens, page, kc, vc, n_pages, scale, B, Hq,
                                                            Hkv, D, parts, parts_bytes, c.stream);
      if (rc) return rc;
      *what = "aq_gemv_w8a8_decode_attn";
      rc = lib.aq_gemv_w8a8_decode_attn(reinterpret_cast<const float*>(parts), lib.aq_paged_attn_decode_slices(total), D, o.w, o.s, o.b.p,
                                        o.b.code, in, x1, AQ_BF16, M, o.N, o.K, c.stream);
    } else {
      void* ws = parts_bytes ? parts : nullptr;
      rc = qk_norm ? lib.aq_rope_paged_attn_decode_qknorm(q, fr, fr_stride, table, P, total, lens, page, kc, vc, n_pages, scale, att, B, Hq,
                                                          Hkv, D, qn.p, kn.p, qn.eps, ws, parts_bytes, c.stream)
                   : lib.aq_rope_paged_attn_decode(q, fr, fr_stride, table, P, total, lens, page, kc, vc, n_pages, scale, att, B, Hq, Hkv,
                                                   D, ws, parts_bytes, c.stream);
      if (rc) return rc;
      rc = projected(o, att, in, x1, codes);
    }
  } else {
    char *qr = base + this->q, *kr = direct ? base + k : nullptr;
    const void *qg = qk_norm ? qn.p : nullptr, *kg = qk_norm ? kn.p : nullptr;
    const bool late = rotates();
    *what = "aq_rope_kv_write";
    rc = late ? lib.aq_rope_kv_cache_write(q, fr, fr_stride, table, P, total - S, S, page, kc, vc, n_pages, kr, B, Hq, Hkv, D, kg, qn.eps,
                                           c.stream)
         : qk_norm ? lib.aq_rope_kv_write_qknorm(q, fr, fr_stride, table, P, total - S, S, page, kc, vc, n_pages, qr, kr, B, Hq, Hkv, D, qg,
                                                 kg, qn.eps, c.stream)
                   : lib.aq_rope_kv_write(q, fr, fr_stride, table, P, total - S, S, page, kc, vc, n_pages, qr, kr, B, Hq, Hkv, D, c.stream);
    if (rc) return rc;
    // what streams behind attention, which itself leaves HBM idle
    const aq_span ahead[3] = {{o.w, o.N * o.K}, {ug.w, ug.N * ug.K}, {down.w, down.N * down.K}};
    if (direct) {
      *what = "aq_prefill_attn_causal";
      const char* v = q + 2 * (A + KV);
      rc = late ? lib.aq_rope_prefill_attn_causal_ahead(q, W, fr, fr_stride, qg, qn.eps, kr, KV, v, W, att, scale, B, S, Hq, Hkv, D, ahead,
                                                        3, c.stream)
                : lib.aq_prefill_attn_causal_ahead(qr, A, kr, KV, v, W, att, scale, B, S, Hq, Hkv, D, ahead, 3, c.stream);
    } else {
      *what = "aq_prefill_attn_paged";
      rc = late ? lib.aq_rope_prefill_attn_paged_ahead(q, W, fr, fr_stride, qg, qn.eps, kc, vc, table, P, total - S, page, n_pages, att,
                                                       scale, B, S, Hq, Hkv, D, ahead, 3, c.stream)
                : lib.aq_prefill_attn_paged_ahead(qr, A, kc, vc, table, P, total - S, page, n_pages, att, scale, B, S, Hq, Hkv, D, ahead, 3,
                                                  c.stream);
    }
    if (rc) return rc;
    rc = projected(o, att, in, x1, codes);
  }
  if (rc) return rc;

  char *h = base + up_gate, *hq = base + h_codes;
  if (swiglu_gemv) {
    *what = "aq_gemv_w8a8_decode_swiglu";
    rc = lib.aq_gemv_w8a8_decode_swiglu(x1, AQ_BF16, n2.p, n2.eps, ug.w, ug.s, ug.b.p, ug.b.code, h, AQ_BF16, M, F, dim, c.stream);
    return rc ? rc : projected(down, h, x1, out, h_codes);
  }
  rc = normed(ug, n2, x1, h, h_codes);
  if (rc) return rc;
  *what = "aq_swiglu_quant_rowwise_i8";
  rc = lib.aq_swiglu_quant_rowwise_i8(h, AQ_BF16, M, F, 2 * F, reinterpret_cast<int8_t*>(hq), sx, c.stream);
  if (rc) return rc;
  *what = few ? "aq_gemv_w8a8_codes" : "aq_linear_w8a8";
  return few ? lib.aq_gemv_w8a8_codes_residual(reinterpret_cast<const int8_t*>(hq), sx, down.w, down.s, down.b.p, down.b.code, x1, out,
                                               AQ_BF16, M, dim, F, c.stream)
             : lib.aq_linear_w8a8_residual(reinterpret_cast<const int8_t*>(hq), sx, down.w, down.s, down.b.p, down.b.code, x1, out,
                                           AQ_BF16, M, dim, F, c.stream);
}

// block_forward(block, x, rotary, cache) -> the block's output, or None where the step-by-step path has to serve
PyObject* block_forward(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS AQ_ARGS(4);
  if (!types.block_ops || !unobserved(types.block_ops)) return none();
  Block b;
  if (!b.read(args[0], args[1], args[2], args[3])) return none();
  b.lay_out();
  Tensor y = b.c.empty({b.B, b.S, b.dim}, ScalarType::BFloat16), mem = b.c.empty({static_cast<int64_t>(b.most)}, ScalarType::Byte);
  const char* what = "";
  const int rc = queued(
      [&] { return b.queue(b.hold_x.const_data_ptr(), y.mutable_data_ptr(), static_cast<char*>(mem.mutable_data_ptr()), &what); });
  return rc ? fail(rc, what) : THPVariable_Wrap(y);
  END_HANDLE_TH_ERRORS
}

// set_block_types(RMSNorm, GQA, MLP, PagedKV, {class: what it defines}, {name: operator or limit as defined}, (limits of
//                 attn_gemv_fusable), {dtype: longest row the norm takes}, {dtype: longest row the activation takes})
PyObject* set_block_types(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  AQ_ARGS(9);
  if (!PyDict_Check(args[4]) || !take_class(args[4], args[1], &types.gqa) || !take_class(args[4], args[2], &types.mlp) ||
      !take_class(args[4], args[3], &types.paged_kv) || !PyDict_Check(args[5]) || !PyDict_Check(args[7]) || !PyDict_Check(args[8]) ||
      !limits_of(args[6], {&types.merge.rows, &types.merge.width, &types.merge.slices, &types.merge.slice, &types.merge.work}))
    return PyErr_Format(PyExc_TypeError, "set_block_types");
  for (int i : {0, 5, 7, 8}) Py_INCREF(args[i]);  // for the life of the process
  types.rms_norm = args[0], types.block_ops = args[5], types.norm_max_k = args[7], types.swiglu_max_f = args[8];
  Py_RETURN_NONE;
}

// bind(handle): take the entry points from the library that ctypes has loaded (CDLL._handle)
PyObject* bind(PyObject*, PyObject* handle) {
  void* h = PyLong_AsVoidPtr(handle);
  if (!h) return PyErr_Occurred() ? nullptr : PyErr_Format(PyExc_ValueError, "null library handle");
  Library l;
#define X(name)                                                  \
  l.name = reinterpret_cast<decltype(l.name)>(dlsym(h, #name));  \
  if (!l.name) return PyErr_Format(PyExc_RuntimeError, "the library lacks " #name);
  AQ_HOST_SYMBOLS(X)
#undef X
  lib = l;
  Py_RETURN_NONE;
}

#define AQ_METHOD(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(name)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {
    {"bind", bind, METH_O, nullptr},
    AQ_METHOD(set_linear_types),
    AQ_METHOD(set_block_types),
    AQ_METHOD(attn_gemv_fusable),
    {"serve_calls", serve_calls, METH_O, nullptr},
    AQ_METHOD(quant_rowwise_i8),
    AQ_METHOD(rmsnorm_quant_rowwise_i8),
    AQ_METHOD(swiglu_quant_rowwise_i8),
    AQ_METHOD(gemv_w8a8_decode),
    AQ_METHOD(gemv_w8a8_codes),
    AQ_METHOD(linear_w8a8),
    AQ_METHOD(quant_tensor_fp8),
    AQ_METHOD(gemv_fp8_decode),
    AQ_METHOD(linear_fp8),
    AQ_METHOD(block_forward),
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", "Native host path of the operators and the fused block.", -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__host() {
  static const struct {
    PyObject** key;
    const char* name;
  } keys[] = {{&k_modules, "_modules"},       {&k_buffers, "_buffers"},         {&k_parameters, "_parameters"},
              {&k_qweight, "qweight"},        {&k_w_scale, "w_scale"},          {&k_bias, "bias"},
              {&k_weight, "weight"},          {&k_norm_eps, "norm_eps"},        {&k_forward, "forward"},
              {&k_fwd_hooks, "_forward_hooks"}, {&k_fwd_pre_hooks, "_forward_pre_hooks"}, {&k_compiled, "_compiled_call_impl"},
              {&k_attention, "attention"},    {&k_mlp, "mlp"},                  {&k_input_norm, "input_norm"},
              {&k_post_norm, "post_attention_norm"}, {&k_qkv, "_qkv"},          {&k_upgate, "_upgate"},
              {&k_o_proj, "o_proj"},          {&k_down, "down"},                {&k_q_norm, "q_norm"},
              {&k_k_norm, "k_norm"},          {&k_decode_attention, "_decode_attention"}, {&k_use_qk_norm, "use_qk_norm"},
              {&k_use_gate, "use_gated_attention"}, {&k_n_heads, "n_heads"},    {&k_n_kv_heads, "n_kv_heads"},
              {&k_head_dim, "head_dim"},      {&k_layer_id, "layer_id"},        {&k_swiglu_quant, "_swiglu_quant"},
              {&k_norm_quant, "_norm_quant"}, {&k_residual_adds, "_residual_adds"}, {&k_k_layers, "k_layers"},
              {&k_v_layers, "v_layers"},      {&k_page_table, "page_table"},    {&k_total_len, "total_len"},
              {&k_seq_lens, "seq_lens"},      {&k_invalid, "_invalid"},         {&k_page_size, "page_size"},
              {&k_shared, "_shared"},         {&k_residual, "residual"},        {&k_norm, "norm"},
              {&k_call, "__call__"},          {&k_decode_rows, "DECODE_MAX_ROWS"},
              {&k_forward_codes, "forward_codes"}, {&k_forward_attn, "forward_attn"}};
  for (const auto& k : keys)
    if (!(*k.key = PyUnicode_InternFromString(k.name))) return nullptr;
  return PyModule_Create(&module);
}
