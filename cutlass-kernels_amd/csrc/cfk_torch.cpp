// The calls of fmha.py on torch tensors, as native code: checks, result tensor, parameter block and launch without the interpreter between
// them.  What bounds the smallest calls is the host: 6.3 us a gemm() of 256 x 256 x 192, of which the launch itself 3.1 to 3.7.  A function
// here answers None, with nothing done, for whatever is not plain -- other types, shapes that do not match, tensors that
// stand for others, torch's function modes -- and the caller goes on in Python, where the errors are raised.
// us a call among others, in Python -> here: gemm() of 256 x 256 x 192 6.3 -> 4.7, of 1024 x 1024 x 1024, which the kernel bounds then, 6.8 -> 6.4;
// fmha_forward() of 4 heads, 256 x 256, D=64 6.0 -> 4.6; where two kernels run, the host is ahead of them either way (10.7 -> 9.9 of 13.2).
#include <Python.h>

#include <cfloat>
#include <cmath>

#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/core/Tensor.h>
#include <ATen/ops/empty_like.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/object_ptr.h>

#include "../../include/cfk_fmha.h"

namespace {

// the library's entry points, as fmha.py has loaded them
struct {
  int64_t (*fmha)(const cfk_fmha_fwd_params *, void *);
  int (*fmha_ws)(const cfk_fmha_fwd_params *, void *, int64_t, void *);
  int (*gemm)(const cfk_gemm_params *, void *);
} api;

// A tensor of the GPU that is nothing but its memory, contiguous: no subclass, no transform's wrapper, no zero or conjugate view.
const at::Tensor *plain(PyObject *x) {
  if (!THPVariable_CheckExact(x)) return nullptr;
  const at::Tensor &t = THPVariable_Unpack(x);
  constexpr c10::DispatchKeySet kPlain = c10::DispatchKeySet({c10::DispatchKey::Dense, c10::DispatchKey::CUDA, c10::DispatchKey::ADInplaceOrView, c10::DispatchKey::AutocastCUDA}) | c10::autograd_dispatch_keyset;
  const uint64_t keys = t.key_set().raw_repr(), gpu = c10::DispatchKeySet(c10::DispatchKey::CUDA).raw_repr();   // (functionalities and backend, a bit each)
  if ((keys & gpu) != gpu || (keys & ~kPlain.raw_repr()) != 0) return nullptr;
  return t.defined() && !t.unsafeGetTensorImpl()->has_symbolic_sizes_strides() && t.is_contiguous() ? &t : nullptr;
}

bool number(PyObject *x, float *f) {   // Python's own numbers that a float holds (struct.pack takes more, and answers for what is beyond)
  if (!PyFloat_CheckExact(x) && !PyLong_CheckExact(x)) return false;
  const double d = PyFloat_AsDouble(x);
  if (d == -1.0 && PyErr_Occurred()) return PyErr_Clear(), false;
  if (std::isfinite(d) && std::fabs(d) > FLT_MAX) return false;
  return *f = (float)d, true;
}

bool choice(PyObject *x, int32_t *i) {
  if (!PyLong_CheckExact(x)) return false;
  const long v = PyLong_AsLong(x);
  if (v == -1 && PyErr_Occurred()) return PyErr_Clear(), false;
  return *i = (int32_t)v, v == 0 || v == 1;
}

bool fits(std::initializer_list<int64_t> sizes) {
  for (int64_t s : sizes)
    if (s > INT32_MAX) return false;
  return true;
}

// gemm(a, b, c, alpha, beta, out, layout): the result; an error code; or None
PyObject *gemm(PyObject *, PyObject *const *args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  cfk_gemm_params p{};
  if (n != 7 || at::impl::torch_function_mode_enabled()) Py_RETURN_NONE;
  const at::Tensor *a = plain(args[0]), *b = a ? plain(args[1]) : nullptr;
  if (!b || !number(args[3], &p.alpha) || !number(args[4], &p.beta) || !choice(args[6], &p.layout)) Py_RETURN_NONE;
  const auto type = a->scalar_type();
  if ((type != at::kHalf && type != at::kFloat) || b->scalar_type() != type) Py_RETURN_NONE;
  const int64_t dims = a->dim();
  if ((dims != 2 && dims != 3) || b->dim() != dims) Py_RETURN_NONE;
  const bool tn = p.layout == CFK_GEMM_TN;
  const int64_t L = dims == 3 ? a->size(0) : 1, M = a->size(-2), K = a->size(-1), N = b->size(tn ? -2 : -1);
  if (b->size(tn ? -1 : -2) != K || (dims == 3 && b->size(0) != L) || !fits({L, M, N, K})) Py_RETURN_NONE;
  const at::Tensor *c = nullptr, *out = nullptr;
  const auto result = [&](PyObject *x, const at::Tensor **t) {   // None, or a tensor like the result
    if (x == Py_None) return true;
    *t = plain(x);
    return *t && (*t)->scalar_type() == type && (*t)->dim() == dims && (*t)->size(-2) == M && (*t)->size(-1) == N && (dims == 2 || (*t)->size(0) == L);
  };
  if (!result(args[2], &c) || !result(args[5], &out)) Py_RETURN_NONE;
  at::Tensor made;
  if (!out) {
    made = dims == 3 ? a->new_empty({L, M, N}) : a->new_empty({M, N});
    out = &made;
  }
  p.dtype = type == at::kHalf ? CFK_FP16 : CFK_FP32;
  p.m = (int32_t)M, p.n = (int32_t)N, p.k = (int32_t)K, p.batch = (int32_t)L;
  p.a = a->data_ptr(), p.b = b->data_ptr(), p.c = c ? c->data_ptr() : nullptr, p.d = out->data_ptr();
  void *stream = c10::hip::getCurrentHIPStream().stream();
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = api.gemm(&p, stream);
  Py_END_ALLOW_THREADS
  if (rc != CFK_OK) return PyLong_FromLong(rc);
  if (made.defined()) return THPVariable_Wrap(std::move(made));
  Py_INCREF(args[5]);
  return args[5];
  END_HANDLE_TH_ERRORS
}

// fmha(q, k, v, o, softmax_scale, q_descale, k_descale, v_descale, v_layout, workspace): the same; workspace(bytes, stream) gives scratch memory or None
PyObject *fmha(PyObject *, PyObject *const *args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  cfk_fmha_fwd_params p{};
  if (n != 10 || at::impl::torch_function_mode_enabled()) Py_RETURN_NONE;
  const at::Tensor *q = plain(args[0]), *k = q ? plain(args[1]) : nullptr, *v = k ? plain(args[2]) : nullptr;
  if (!v || q->dim() != 4 || k->dim() != 4 || v->dim() != 4) Py_RETURN_NONE;
  if (!number(args[5], &p.q_descale) || !number(args[6], &p.k_descale) || !number(args[7], &p.v_descale) || !choice(args[8], &p.v_layout)) Py_RETURN_NONE;
  const auto type = q->scalar_type(), v_type = v->scalar_type();
  if ((type != at::kHalf && type != at::kFloat8_e4m3fn && type != at::kByte) || k->scalar_type() != type || (v_type != type && v_type != at::kHalf)) Py_RETURN_NONE;
  const int64_t B = q->size(0), Sq = q->size(1), H = q->size(2), D = q->size(3), Skv = k->size(1);
  if (k->size(0) != B || k->size(2) != H || k->size(3) != D || !fits({B, Sq, H, D, Skv}) || D == 0) Py_RETURN_NONE;
  if (p.v_layout == CFK_V_BSHD ? v->sizes() != k->sizes() : v->sizes() != at::IntArrayRef({B, D, H, Skv})) Py_RETURN_NONE;
  if (args[4] == Py_None) p.softmax_scale = (float)(1.0 / std::sqrt((double)D));
  else if (!number(args[4], &p.softmax_scale)) Py_RETURN_NONE;
  const at::Tensor *o = nullptr;
  at::Tensor made;
  if (args[3] != Py_None) {
    o = plain(args[3]);
    if (!o || o->scalar_type() != at::kHalf || o->sizes() != q->sizes()) Py_RETURN_NONE;
  } else {
    made = at::empty_like(*q, q->options().dtype(at::kHalf));
    o = &made;
  }
  p.dtype = type == at::kHalf ? CFK_FP16 : CFK_FP8_E4M3;
  p.v_dtype = v_type == type ? p.dtype : CFK_FP16;
  p.batch = (int32_t)B, p.heads = (int32_t)H, p.seqlen_q = (int32_t)Sq, p.seqlen_kv = (int32_t)Skv, p.head_dim = (int32_t)D;
  p.q = q->data_ptr(), p.k = k->data_ptr(), p.v = v->data_ptr(), p.o = o->data_ptr();
  void *stream = c10::hip::getCurrentHIPStream().stream();
  int64_t rc;
  Py_BEGIN_ALLOW_THREADS
  rc = api.fmha(&p, stream);
  Py_END_ALLOW_THREADS
  if (rc > 0) {   // the call is not made yet: it can use this much scratch memory
    THPObjectPtr ws(PyObject_CallFunction(args[9], "LK", (long long)rc, (unsigned long long)(uintptr_t)stream));
    if (!ws) return nullptr;
    void *scratch = nullptr;
    if (ws.get() != Py_None) {
      THPObjectPtr address(PyObject_CallMethod(ws.get(), "data_ptr", nullptr));
      if (!address) return nullptr;
      scratch = PyLong_AsVoidPtr(address.get());
      if (!scratch && PyErr_Occurred()) return nullptr;
    }
    const int64_t bytes = rc;
    Py_BEGIN_ALLOW_THREADS
    rc = api.fmha_ws(&p, scratch, bytes, stream);
    Py_END_ALLOW_THREADS
  }
  if (rc != CFK_OK) return PyLong_FromLong((long)rc);
  if (made.defined()) return THPVariable_Wrap(std::move(made));
  Py_INCREF(args[3]);
  return args[3];
  END_HANDLE_TH_ERRORS
}

// setup(addresses of cfk_fmha_forward_or_workspace, cfk_fmha_forward_ws and cfk_gemm)
PyObject *setup(PyObject *, PyObject *args) {
  unsigned long long f, w, g;
  if (!PyArg_ParseTuple(args, "KKK", &f, &w, &g)) return nullptr;
  api = {(decltype(api.fmha))f, (decltype(api.fmha_ws))w, (decltype(api.gemm))g};
  Py_RETURN_NONE;
}

PyMethodDef methods[] = {{"setup", setup, METH_VARARGS, nullptr},
                         {"gemm", (PyCFunction)(void (*)(void))gemm, METH_FASTCALL, nullptr},
                         {"fmha", (PyCFunction)(void (*)(void))fmha, METH_FASTCALL, nullptr},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "cfk_torch", nullptr, -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit_cfk_torch(void) {
  PyObject *m = PyModule_Create(&module);
  if (m && PyModule_AddStringConstant(m, "torch_version", CFK_TORCH_VERSION) == 0) return m;   // (torch's C++ interface holds for one version)
  Py_XDECREF(m);
  return nullptr;
}
