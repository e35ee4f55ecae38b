// Launches of the forward and backward from torch tensors (CPython extension
// pallas_flexattn/_launch.so): outputs and workspace allocated, operands made
// dense and the C ABI called without going through Python objects and ctypes
// conversions for every pointer.  Host code only; the C ABI's entry points are
// handed over by address (bind), so it links against torch alone.
//
// Why: a small training step is bound by the host.  At B2 H4 S300 D64 the
// Python form of these two calls took 13 us (forward) and 18 us (backward; about
// 34 on the autograd engine's thread) of a 136 us step whose kernels take 40.
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <ATen/ATen.h>

#include <cstdint>

namespace {

using fwd_fn = int (*)(const void*, const void*, const void*, const void*, void*, float*, void*);
using bwd_fn = int (*)(const void*, const void*, const void*, const void*, const void*, const float*, const void*,
                       void*, void*, void*, void*, size_t, void*);
using ws_fn = size_t (*)(const void*);

fwd_fn g_fwd = nullptr;
bwd_fn g_bwd = nullptr;
ws_fn g_bwd_ws = nullptr;

void* address(PyObject* x) { return PyLong_AsVoidPtr(x); }

// Contiguous with a 16-byte aligned base (the kernels use 16-byte loads).
at::Tensor dense16(const at::Tensor& t) {
  at::Tensor c = t.contiguous();
  return (reinterpret_cast<uintptr_t>(c.const_data_ptr()) & 15) ? c.clone() : c;
}

const at::Tensor* tensor(PyObject* x) {
  if (!THPVariable_Check(x)) {
    PyErr_SetString(PyExc_TypeError, "expected a torch tensor");
    return nullptr;
  }
  return &THPVariable_Unpack(x);
}

// bind(fa_fwd, fa_bwd_split, fa_bwd_split_workspace_bytes)
PyObject* py_bind(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 3) {
    PyErr_SetString(PyExc_TypeError, "bind takes 3 addresses");
    return nullptr;
  }
  g_fwd = reinterpret_cast<fwd_fn>(address(a[0]));
  g_bwd = reinterpret_cast<bwd_fn>(address(a[1]));
  g_bwd_ws = reinterpret_cast<ws_fn>(address(a[2]));
  if (PyErr_Occurred()) return nullptr;
  Py_RETURN_NONE;
}

// fwd(params, q, k, v, stream) -> (status, o, lse).  The caller has checked
// q, k, v against each other and against the params.
PyObject* py_fwd(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 5 || !g_fwd) {
    PyErr_SetString(PyExc_TypeError, "fwd(params, q, k, v, stream) after bind");
    return nullptr;
  }
  const void* params = address(a[0]);
  void* stream = address(a[4]);
  if (PyErr_Occurred()) return nullptr;
  const at::Tensor* t[3];
  for (int i = 0; i < 3; ++i)
    if (!(t[i] = tensor(a[1 + i]))) return nullptr;
  const at::Tensor q = dense16(*t[0]), k = dense16(*t[1]), v = dense16(*t[2]);
  at::Tensor o = at::empty_like(q);
  at::Tensor lse = at::empty(q.sizes().slice(0, 3), q.options().dtype(at::kFloat));
  const void *qp = q.const_data_ptr(), *kp = k.const_data_ptr(), *vp = v.const_data_ptr();
  void* op = o.mutable_data_ptr();
  float* lp = lse.mutable_data_ptr<float>();
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = g_fwd(params, qp, kp, vp, op, lp, stream);
  Py_END_ALLOW_THREADS
  return Py_BuildValue("iNN", rc, THPVariable_Wrap(o), THPVariable_Wrap(lse));
  END_HANDLE_TH_ERRORS
}

// bwd(params, q, k, v, o, lse, do, stream) -> (status, dq, dk, dv)
PyObject* py_bwd(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 8 || !g_bwd) {
    PyErr_SetString(PyExc_TypeError, "bwd(params, q, k, v, o, lse, do, stream) after bind");
    return nullptr;
  }
  const void* params = address(a[0]);
  void* stream = address(a[7]);
  if (PyErr_Occurred()) return nullptr;
  const at::Tensor* t[6];
  for (int i = 0; i < 6; ++i)
    if (!(t[i] = tensor(a[1 + i]))) return nullptr;
  const at::Tensor q = dense16(*t[0]), k = dense16(*t[1]), v = dense16(*t[2]), o = dense16(*t[3]);
  const at::Tensor lse = t[4]->scalar_type() == at::kFloat ? t[4]->contiguous() : t[4]->to(at::kFloat).contiguous();
  const at::Tensor dout = dense16(t[5]->scalar_type() == q.scalar_type() ? *t[5] : t[5]->to(q.scalar_type()));
  if (o.sizes() != q.sizes() || dout.sizes() != q.sizes() || lse.sizes() != q.sizes().slice(0, 3) ||
      o.scalar_type() != q.scalar_type()) {
    PyErr_SetString(PyExc_ValueError, "o / do / lse shapes do not match q");
    return nullptr;
  }
  if (o.device() != q.device() || dout.device() != q.device() || lse.device() != q.device()) {
    PyErr_SetString(PyExc_ValueError, "o / do / lse are not on q's device");
    return nullptr;
  }
  const size_t need = g_bwd_ws(params), bytes = need < 256 ? 256 : need;
  at::Tensor ws = at::empty({static_cast<int64_t>(bytes)}, q.options().dtype(at::kByte));
  at::Tensor dq = at::empty_like(q), dk = at::empty_like(k), dv = at::empty_like(v);
  const void *qp = q.const_data_ptr(), *kp = k.const_data_ptr(), *vp = v.const_data_ptr(), *op = o.const_data_ptr(),
             *dp = dout.const_data_ptr();
  const float* lp = lse.const_data_ptr<float>();
  void *gq = dq.mutable_data_ptr(), *gk = dk.mutable_data_ptr(), *gv = dv.mutable_data_ptr(), *wp = ws.mutable_data_ptr();
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = g_bwd(params, qp, kp, vp, op, lp, dp, gq, gk, gv, wp, bytes, stream);
  Py_END_ALLOW_THREADS
  return Py_BuildValue("iNNN", rc, THPVariable_Wrap(dq), THPVariable_Wrap(dk), THPVariable_Wrap(dv));
  END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {
    {"bind", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(py_bind)), METH_FASTCALL, nullptr},
    {"fwd", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(py_fwd)), METH_FASTCALL, nullptr},
    {"bwd", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(py_bwd)), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_launch", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__launch(void) { return PyModule_Create(&module); }
