// The operators' usual calls without the Python in between: device tensors in, a fresh tensor out. A small operator's time is the
// host's (a layer norm of 512 x 768: 11.9 us a call, 3.4 of them the launch, 1.7 the output's allocation, the rest Python and
// ctypes; 4.9 this way). Each function takes the arguments of its namesake in hexmi/ops.py and returns the result, or None for a
// call that is not of the plain form -- host tensors, other types, strides, shapes that do not fit, subclasses, an active
// tracing or functorch mode, another device than the current one -- which ops.py then handles (and refuses) as ever. Built against
// torch's own headers; calls the C ABI of include/hexmi.h.
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cmath>
#include <cstddef>

#include "hexmi.h"

namespace {

PyObject* g_check = nullptr;                       // hexmi._lib.check: raises for a status

// A tensor as this module takes it: torch.Tensor or Parameter itself, dense in device memory, no wrapper of any kind.
const at::Tensor* dense(PyObject* o) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || !t.has_storage() || t.numel() == 0) return nullptr;
  static const c10::DispatchKeySet other({c10::DispatchKey::Python, c10::DispatchKey::Conjugate, c10::DispatchKey::Negative,
                                          c10::DispatchKey::ZeroTensor, c10::DispatchKey::FuncTorchBatched,
                                          c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::Functionalize});
  if (t.unsafeGetTensorImpl()->key_set().has_any(other)) return nullptr;
  return &t;
}
const at::Tensor* contiguous(PyObject* o) {
  const at::Tensor* t = dense(o);
  return t && t->is_contiguous() ? t : nullptr;
}
bool modes_active() {
  return c10::impl::TorchDispatchModeTLS::any_modes_set() || at::impl::torch_function_mode_enabled() ||
         c10::impl::tls_local_dispatch_key_set().included_.has(c10::DispatchKey::FuncTorchDynamicLayerFrontMode);
}
int code_of(at::ScalarType s) {
  return s == at::kHalf ? HEXMI_F16 : s == at::kFloat ? HEXMI_F32 : s == at::kBFloat16 ? HEXMI_BF16 : 0;
}

// The current stream if the tensor is on the current device.
struct Launch {
  hipStream_t stream = nullptr;
  bool ok = false;
  explicit Launch(const at::Tensor& t) {
    if (modes_active()) return;
    const c10::hip::HIPStream s = c10::hip::getCurrentHIPStream();
    ok = s.device_index() == t.device().index();
    stream = s.stream();
  }
};
at::Tensor fresh(at::IntArrayRef sizes, at::ScalarType type, const at::Tensor& like) {
  return at::Tensor(at::detail::empty_cuda(sizes, type, like.device(), c10::nullopt));
}
// an operand is only read: a copy-on-write one stays shared
const void* in(const at::Tensor* t) { return t ? t->const_data_ptr() : nullptr; }

// an operand that may be None: true if absent or plain, of `sizes` and `type` beside `like`
bool optional(PyObject* o, const at::Tensor*& t, at::IntArrayRef sizes, at::ScalarType type, const at::Tensor& like) {
  t = nullptr;
  if (o == Py_None) return true;
  t = contiguous(o);
  return t && t->scalar_type() == type && t->sizes() == sizes && t->device() == like.device();
}
bool number(PyObject* o, double& v) {
  if (!PyFloat_CheckExact(o) && !PyLong_CheckExact(o)) return false;
  v = PyFloat_AsDouble(o);
  if (v == -1.0 && PyErr_Occurred()) {
    PyErr_Clear();
    return false;
  }
  return true;
}
bool flag(PyObject* o, bool& v) {
  if (o != Py_True && o != Py_False) return false;
  v = o == Py_True;
  return true;
}

PyObject* finish(int status, const char* what, at::Tensor&& out) {
  if (status != HEXMI_OK) {
    PyObject* r = g_check ? PyObject_CallFunction(g_check, "is", status, what) : nullptr;
    Py_XDECREF(r);
    if (!PyErr_Occurred()) PyErr_Format(PyExc_RuntimeError, "%s failed with status %d", what, status);
    return nullptr;
  }
  return THPVariable_Wrap(std::move(out));
}

// C++ exceptions (the allocator out of memory among them) become Python's
template <typename F>
PyObject* guarded(F&& f) {
  HANDLE_TH_ERRORS
  return f();
  END_HANDLE_TH_ERRORS
}
#define HEXMI_NOT_PLAIN Py_RETURN_NONE
// f(a...) without the interpreter lock, which is back before anything leaves this function. The arguments, pointers of tensors that
// other threads may hold too, are taken under the lock.
template <typename... P, typename... A>
int unlocked(int (*f)(P...), A... a) {
  PyThreadState* state = PyEval_SaveThread();
  int status;
  try {
    status = f(static_cast<P>(a)...);
  } catch (...) {
    PyEval_RestoreThread(state);
    throw;
  }
  PyEval_RestoreThread(state);
  return status;
}

struct Rows {
  const at::Tensor* x;
  int code;
  int64_t rows, cols;
  bool set(PyObject* o) {
    x = contiguous(o);
    if (!x || x->dim() < 1) return false;
    code = code_of(x->scalar_type());
    cols = x->size(-1);
    rows = x->numel() / cols;
    return code != 0;
  }
  // scratch of the split forms, empty where they are not taken
  at::Tensor scratch(int64_t& bytes) const {
    bytes = hexmi_row_workspace(rows, cols, 0, code);
    return bytes ? fresh({bytes}, at::kByte, *x) : at::Tensor();
  }
};

// softmax(x)
PyObject* softmax(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    Rows r;
    if (n != 1 || !r.set(a[0])) HEXMI_NOT_PLAIN;
    const Launch at(*r.x);
    if (!at.ok) HEXMI_NOT_PLAIN;
    at::Tensor out = fresh(r.x->sizes(), r.x->scalar_type(), *r.x);
    int64_t bytes;
    const at::Tensor ws = r.scratch(bytes);
    return finish(unlocked(hexmi_softmax_ws, in(r.x), out.mutable_data_ptr(), r.rows, r.cols, r.cols, r.cols, 0, r.code,
                           bytes ? ws.mutable_data_ptr() : nullptr, bytes, at.stream), "hexmi_softmax_ws", std::move(out));
  });
}

// rms_norm(x, weight or None, eps)
PyObject* rms_norm(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    Rows r;
    const at::Tensor* w;
    double eps;
    if (n != 3 || !r.set(a[0]) || !optional(a[1], w, {r.cols}, r.x->scalar_type(), *r.x) || !number(a[2], eps)) HEXMI_NOT_PLAIN;
    const Launch at(*r.x);
    if (!at.ok) HEXMI_NOT_PLAIN;
    at::Tensor out = fresh(r.x->sizes(), r.x->scalar_type(), *r.x);
    int64_t bytes;
    const at::Tensor ws = r.scratch(bytes);
    return finish(unlocked(hexmi_rms_norm_ws, in(r.x), in(w), out.mutable_data_ptr(), r.rows, r.cols, r.cols, r.cols, (float)eps, 0,
                           r.code, bytes ? ws.mutable_data_ptr() : nullptr, bytes, at.stream), "hexmi_rms_norm_ws", std::move(out));
  });
}

// layer_norm(x, weight or None, bias or None, eps)
PyObject* layer_norm(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    Rows r;
    const at::Tensor *w, *b;
    double eps;
    if (n != 4 || !r.set(a[0]) || !optional(a[1], w, {r.cols}, r.x->scalar_type(), *r.x) ||
        !optional(a[2], b, {r.cols}, r.x->scalar_type(), *r.x) || !number(a[3], eps)) HEXMI_NOT_PLAIN;
    const Launch at(*r.x);
    if (!at.ok) HEXMI_NOT_PLAIN;
    at::Tensor out = fresh(r.x->sizes(), r.x->scalar_type(), *r.x);
    int64_t bytes;
    const at::Tensor ws = r.scratch(bytes);
    return finish(unlocked(hexmi_layer_norm_ws, in(r.x), in(w), in(b), out.mutable_data_ptr(), nullptr, nullptr, r.rows, r.cols, r.cols,
                           r.cols, (float)eps, 0, r.code, bytes ? ws.mutable_data_ptr() : nullptr, bytes, at.stream),
                  "hexmi_layer_norm_ws", std::move(out));
  });
}

// matmul(a, b, trans_b, bias or None, residual or None), result of the operands' type
PyObject* matmul(PyObject*, PyObject* const* v, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    const at::Tensor* a = n == 5 ? contiguous(v[0]) : nullptr;
    const at::Tensor* b = a ? contiguous(v[1]) : nullptr;
    bool tb;
    if (!b || !flag(v[2], tb) || a->dim() != 2 || b->dim() != 2 || a->scalar_type() != b->scalar_type() || a->device() != b->device())
      HEXMI_NOT_PLAIN;
    const int code = code_of(a->scalar_type());
    const int64_t M = a->size(0), K = a->size(1), N = b->size(tb ? 0 : 1);
    const at::Tensor *bias, *res;
    if (!code || b->size(tb ? 1 : 0) != K || !optional(v[3], bias, {N}, a->scalar_type(), *a) ||
        !optional(v[4], res, {M, N}, a->scalar_type(), *a)) HEXMI_NOT_PLAIN;
    const Launch at(*a);
    if (!at.ok) HEXMI_NOT_PLAIN;
    at::Tensor out = fresh({M, N}, a->scalar_type(), *a);
    const int64_t bytes = K >= HEXMI_GEMM_ONE_LAUNCH_K ? hexmi_gemm_workspace(M, N, K, code, tb ? 1 : 0) : 0;
    const at::Tensor ws = bytes ? fresh({bytes}, at::kByte, *a) : at::Tensor();
    return finish(unlocked(hexmi_gemm_ws, M, N, K, in(a), K, in(b), tb ? K : N, out.mutable_data_ptr(), N, in(bias), in(res), res ? N : 0,
                           code, code, tb ? 1 : 0, bytes ? ws.mutable_data_ptr() : nullptr, bytes, at.stream), "hexmi_gemm_ws", std::move(out));
  });
}

// w8a16_matmul(a, w, scales, zero_points or None), a scale (and zero point) per channel, no scratch
PyObject* w8a16_matmul(PyObject*, PyObject* const* v, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    const at::Tensor* a = n == 4 ? contiguous(v[0]) : nullptr;
    const at::Tensor* w = a ? contiguous(v[1]) : nullptr;
    if (!w || a->dim() != 2 || w->dim() != 2 || a->scalar_type() != at::kHalf || w->scalar_type() != at::kChar ||
        a->device() != w->device() || a->size(1) != w->size(1)) HEXMI_NOT_PLAIN;
    const int64_t M = a->size(0), K = a->size(1), N = w->size(0);
    const at::Tensor *s, *z;
    if (v[2] == Py_None || !optional(v[2], s, {N}, at::kHalf, *a) || !optional(v[3], z, {N}, at::kChar, *a)) HEXMI_NOT_PLAIN;
    if (!z && hexmi_gemm_w8a16_workspace_helps(M, N, K)) HEXMI_NOT_PLAIN;      // ops.py keeps that scratch
    const Launch at(*a);
    if (!at.ok) HEXMI_NOT_PLAIN;
    at::Tensor out = fresh({M, N}, at::kHalf, *a);
    if (z)
      return finish(unlocked(hexmi_gemm_w8a16_ex, M, N, K, in(a), in(w), in(s), in(z), 0, out.mutable_data_ptr(), at.stream),
                    "hexmi_gemm_w8a16_ex", std::move(out));
    return finish(unlocked(hexmi_gemm_w8a16_ws, M, N, K, in(a), in(w), in(s), out.mutable_data_ptr(), nullptr, 0, at.stream),
                  "hexmi_gemm_w8a16_ws", std::move(out));
  });
}

// flash_attention(q, k, v, sm_scale or None, causal), result of the operands' type
PyObject* flash_attention(PyObject*, PyObject* const* v, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    const at::Tensor *q = n == 5 ? dense(v[0]) : nullptr, *k = q ? dense(v[1]) : nullptr, *w = k ? dense(v[2]) : nullptr;
    bool causal;
    if (!w || !flag(v[4], causal) || q->dim() != 4 || q->sizes() != k->sizes() || q->sizes() != w->sizes() ||
        q->scalar_type() != k->scalar_type() || q->scalar_type() != w->scalar_type() || q->device() != k->device() ||
        q->device() != w->device()) HEXMI_NOT_PLAIN;
    const int code = code_of(q->scalar_type());
    const int64_t Z = q->size(0), H = q->size(1), S = q->size(2), D = q->size(3);
    double scale = 1.0 / std::sqrt((double)D);
    if (!code || (v[3] != Py_None && !number(v[3], scale))) HEXMI_NOT_PLAIN;
    const bool whole = q->is_contiguous() && k->is_contiguous() && w->is_contiguous();
    if (!whole && (q->stride(3) != 1 || k->stride(3) != 1 || w->stride(3) != 1)) HEXMI_NOT_PLAIN;
    const Launch at(*q);
    if (!at.ok) HEXMI_NOT_PLAIN;
    at::Tensor out = fresh(q->sizes(), q->scalar_type(), *q);
    if (whole)
      return finish(unlocked(hexmi_flash_attn_fwd, in(q), in(k), in(w), out.mutable_data_ptr(), Z, H, S, D, (float)scale, causal ? 1 : 0,
                             code, code, at.stream), "hexmi_flash_attn_fwd", std::move(out));
    const int64_t strides[9] = {q->stride(0), q->stride(1), q->stride(2), k->stride(0), k->stride(1), k->stride(2),
                                w->stride(0), w->stride(1), w->stride(2)};
    const int status = unlocked(hexmi_flash_attn_fwd_strided, in(q), in(k), in(w), out.mutable_data_ptr(), Z, H, S, D, strides,
                                (float)scale, causal ? 1 : 0, code, code, at.stream);
    if (status == HEXMI_ENOTSUP) HEXMI_NOT_PLAIN;                            // ops.py copies the operands
    return finish(status, "hexmi_flash_attn_fwd_strided", std::move(out));
  });
}

// attention(q, k, v, mask or None, sm_scale or None), result of the operands' type
PyObject* attention(PyObject*, PyObject* const* v, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    const at::Tensor *q = n == 5 ? contiguous(v[0]) : nullptr, *k = q ? contiguous(v[1]) : nullptr, *w = k ? contiguous(v[2]) : nullptr;
    if (!w || q->dim() != 3 || k->dim() != 3 || w->sizes() != k->sizes() || q->size(0) != k->size(0) || q->size(2) != k->size(2) ||
        q->scalar_type() != k->scalar_type() || q->scalar_type() != w->scalar_type() || q->device() != k->device() ||
        q->device() != w->device()) HEXMI_NOT_PLAIN;
    const int code = code_of(q->scalar_type());
    const int64_t B = q->size(0), Sq = q->size(1), D = q->size(2), Skv = k->size(1);
    const at::Tensor* mask;
    double scale = 1.0 / std::sqrt((double)D);
    if (!code || !optional(v[3], mask, {B, Sq, Skv}, q->scalar_type(), *q) || (v[4] != Py_None && !number(v[4], scale))) HEXMI_NOT_PLAIN;
    const Launch at(*q);
    if (!at.ok) HEXMI_NOT_PLAIN;
    at::Tensor out = fresh(q->sizes(), q->scalar_type(), *q);
    const int64_t bytes = Skv > HEXMI_ATTENTION_ONE_LAUNCH_KEYS ? hexmi_attention_workspace(B, Sq, Skv, D, mask ? 1 : 0, code) : 0;
    const at::Tensor ws = bytes ? fresh({bytes}, at::kByte, *q) : at::Tensor();
    return finish(unlocked(hexmi_attention_ws, in(q), in(k), in(w), in(mask), out.mutable_data_ptr(), B, Sq, Skv, D, (float)scale, code,
                           code, bytes ? ws.mutable_data_ptr() : nullptr, bytes, at.stream), "hexmi_attention_ws", std::move(out));
  });
}

// unary(op number, x)
PyObject* unary(PyObject*, PyObject* const* v, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    const at::Tensor* x = n == 2 ? contiguous(v[1]) : nullptr;
    const int code = x ? code_of(x->scalar_type()) : 0;
    if (!code) HEXMI_NOT_PLAIN;
    const int op = (int)PyLong_AsLong(v[0]);
    const Launch at(*x);
    if (!at.ok) HEXMI_NOT_PLAIN;
    at::Tensor out = fresh(x->sizes(), x->scalar_type(), *x);
    return finish(unlocked(hexmi_unary, op, in(x), out.mutable_data_ptr(), x->numel(), code, at.stream), "hexmi_unary",
                  std::move(out));
  });
}

// binary(op number, a, b)
PyObject* binary(PyObject*, PyObject* const* v, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    const at::Tensor *a = n == 3 ? contiguous(v[1]) : nullptr, *b = a ? contiguous(v[2]) : nullptr;
    const int code = b ? code_of(a->scalar_type()) : 0;
    if (!code || a->sizes() != b->sizes() || a->scalar_type() != b->scalar_type() || a->device() != b->device()) HEXMI_NOT_PLAIN;
    const int op = (int)PyLong_AsLong(v[0]);
    const Launch at(*a);
    if (!at.ok) HEXMI_NOT_PLAIN;
    at::Tensor out = fresh(a->sizes(), a->scalar_type(), *a);
    return finish(unlocked(hexmi_binary, op, in(a), in(b), out.mutable_data_ptr(), a->numel(), code, at.stream), "hexmi_binary",
                  std::move(out));
  });
}

// set_check(f): f(status, what) raises for a status that is not OK
PyObject* set_check(PyObject*, PyObject* f) {
  Py_INCREF(f);
  Py_XSETREF(g_check, f);
  Py_RETURN_NONE;
}

// A function above as an object of a type of its own: dynamo breaks its graph at such a call without a word, at a built-in function's
// with a warning. Called as fast.
typedef PyObject* (*Function)(PyObject*, PyObject* const*, Py_ssize_t);
struct Operator {
  PyObject_HEAD
  vectorcallfunc call;
  Function f;
};
PyObject* call_operator(PyObject* self, PyObject* const* args, size_t n, PyObject* names) {
  if (names && PyTuple_GET_SIZE(names) != 0) {
    PyErr_SetString(PyExc_TypeError, "positional arguments only");
    return nullptr;
  }
  return reinterpret_cast<Operator*>(self)->f(nullptr, args, PyVectorcall_NARGS(n));
}
PyTypeObject g_operator_type = {PyVarObject_HEAD_INIT(nullptr, 0)};
bool add_operator(PyObject* m, const char* name, Function f) {
  Operator* o = PyObject_New(Operator, &g_operator_type);
  if (!o) return false;
  o->call = call_operator;
  o->f = f;
  if (PyModule_AddObject(m, name, reinterpret_cast<PyObject*>(o)) == 0) return true;
  Py_DECREF(o);
  return false;
}

PyMethodDef g_methods[] = {{"set_check", set_check, METH_O, nullptr}, {nullptr, nullptr, 0, nullptr}};
PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_front", "The operators' usual calls, natively.", -1, g_methods};

}  // namespace

// torch_version: what it was built for (HEXMI_TORCH_VERSION, from the build)
PyMODINIT_FUNC PyInit__front() {
  g_operator_type.tp_name = "hexmi._front.Operator";
  g_operator_type.tp_basicsize = sizeof(Operator);
  g_operator_type.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_HAVE_VECTORCALL;
  g_operator_type.tp_vectorcall_offset = offsetof(Operator, call);
  g_operator_type.tp_call = PyVectorcall_Call;
  if (PyType_Ready(&g_operator_type) != 0) return nullptr;
  PyObject* m = PyModule_Create(&g_module);
  if (!m) return nullptr;
#define HEXMI_OPERATOR(f) add_operator(m, #f, f)
  if (!(HEXMI_OPERATOR(softmax) && HEXMI_OPERATOR(rms_norm) && HEXMI_OPERATOR(layer_norm) && HEXMI_OPERATOR(matmul) &&
        HEXMI_OPERATOR(w8a16_matmul) && HEXMI_OPERATOR(flash_attention) && HEXMI_OPERATOR(attention) && HEXMI_OPERATOR(unary) &&
        HEXMI_OPERATOR(binary) && PyModule_AddStringConstant(m, "torch_version", HEXMI_TORCH_VERSION) == 0))
    Py_CLEAR(m);
#undef HEXMI_OPERATOR
  return m;
}
