// fastcall.cpp -- native call path of decodebench_amd.ops (a CPython extension
// module, _fastcall).
//
// One function per op.  It checks the arguments as the Python op does,
// allocates the output, finds the current stream and calls the C ABI entry
// point; whatever it does not take as it is (another device current, a tensor
// subclass, a wrong shape or type, a workspace that has to be made, a non-zero
// status) it answers with None, and the Python op then does the same work, or
// raises, step by step.  In Python those steps took 6.5-7.5 us a call on the
// host of an MI355X, more than the small kernels take on the GPU: F1 [2048,
// 2048] at one row 7.1-7.7 us a call, 5.0 through here; F4 at batch 1, L = 8192
// 10.4 and 8.9.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <climits>
#include <cmath>
#include <cstdint>

#include "../../include/decodebench_hip.h"

#ifndef DB_BUILT_FOR
#error "build with decodebench_amd.build, which defines DB_BUILT_FOR"
#endif

namespace {

struct Abi {
  decltype(&db_f1_rmsnorm_gemv) f1;
  decltype(&db_f2_gateup_swiglu) f2;
  decltype(&db_f2_rmsnorm_gateup_swiglu) f2n;
  decltype(&db_gemv) gemv;
  decltype(&db_f4_default_splits) f4_default_splits;
  decltype(&db_f4_workspace_bytes) f4_workspace_bytes;
  decltype(&db_f4_splitkv) f4;
  decltype(&db_stream_capture_id) capture_id;
  decltype(&db_gemv_workspace_bytes) gemv_workspace_bytes;
  decltype(&db_gemv_ws) gemv_ws;
} abi;

PyObject* raw_stream = nullptr;  // device index -> current stream's handle
PyObject* get_device = nullptr;  // () -> current device
PyObject* workspaces = nullptr;  // dict (device, stream, bytes) -> tensor
PyObject* cu_counts = nullptr;   // dict device -> compute units

const at::Tensor* tensor(PyObject* o) {
  return THPVariable_CheckExact(o) ? &THPVariable_Unpack(o) : nullptr;
}

// A contiguous GPU tensor of the type, on device `idx` (any if -1).
bool plain(const at::Tensor* t, at::ScalarType type, int idx) {
  return t && t->is_cuda() && t->scalar_type() == type && t->is_contiguous() &&
         (idx < 0 || t->get_device() == idx);
}

// The current stream of device `idx` if that is the current device.
// 1: found, 0: another device is current, -1: a Python error is set.
int stream_of(int idx, void** stream) {
  PyObject* d = PyObject_CallNoArgs(get_device);
  if (!d) return -1;
  const long cur = PyLong_AsLong(d);
  if (cur == -1 && PyErr_Occurred()) {
    Py_DECREF(d);
    return -1;
  }
  if (cur != idx) {
    Py_DECREF(d);
    return 0;
  }
  PyObject* s = PyObject_CallFunctionObjArgs(raw_stream, d, nullptr);
  Py_DECREF(d);
  if (!s) return -1;
  *stream = PyLong_AsVoidPtr(s);
  Py_DECREF(s);
  return *stream == nullptr && PyErr_Occurred() ? -1 : 1;
}

bool number(PyObject* o, double* v) {
  if (!PyFloat_CheckExact(o)) return false;
  *v = PyFloat_AS_DOUBLE(o);
  return true;
}

// fp16 weights without a scale, or e4m3 bytes with one fp32 scale per row.
bool weights(const at::Tensor* w, PyObject* scale, int64_t N, int idx, int* dtype,
             const float** sp) {
  *sp = nullptr;
  if (plain(w, at::kHalf, idx)) {
    *dtype = DB_DTYPE_F16;
    return scale == Py_None;
  }
  if (!plain(w, at::kFloat8_e4m3fn, idx) && !plain(w, at::kByte, idx)) return false;
  const at::Tensor* s = tensor(scale);
  if (!plain(s, at::kFloat, idx) || s->dim() != 1 || s->size(0) != N) return false;
  *dtype = DB_DTYPE_FP8_E4M3;
  *sp = static_cast<const float*>(s->data_ptr());
  return true;
}

// A GEMV op of x [B, K] or [K] on w0 (and w1) [N, K]; g and eps in the norm
// modes.  New reference, Py_None where the Python op has to take over.
PyObject* gemv_op(PyObject* xo, PyObject* go, PyObject* w0o, PyObject* w1o, PyObject* epso,
                  PyObject* s0o, PyObject* s1o) {
  const at::Tensor* x = tensor(xo);
  if (!plain(x, at::kHalf, -1)) Py_RETURN_NONE;
  const int64_t dim = x->dim();
  if (dim != 1 && dim != 2) Py_RETURN_NONE;
  const int idx = x->get_device();
  const int64_t B = dim == 2 ? x->size(0) : 1, K = x->size(dim - 1);
  const at::Tensor* w0 = tensor(w0o);
  const at::Tensor* w1 = w1o ? tensor(w1o) : nullptr;
  if (!w0 || w0->dim() != 2 || w0->size(1) != K) Py_RETURN_NONE;
  const int64_t N = w0->size(0);
  if (B > INT_MAX || K > INT_MAX || N > INT_MAX) Py_RETURN_NONE;
  int dtype = 0, dtype1 = 0;
  const float *s0 = nullptr, *s1 = nullptr;
  if (!weights(w0, s0o, N, idx, &dtype, &s0)) Py_RETURN_NONE;
  if (w1o && (!w1 || w1->sizes() != w0->sizes() || w1->scalar_type() != w0->scalar_type() ||
              !weights(w1, s1o, N, idx, &dtype1, &s1)))
    Py_RETURN_NONE;
  const at::Tensor* g = nullptr;
  double eps = 0.0;
  if (go) {
    g = tensor(go);
    if (!plain(g, at::kHalf, idx) || g->dim() != 1 || g->size(0) != K || !number(epso, &eps))
      Py_RETURN_NONE;
  }
  void* stream = nullptr;
  const int found = stream_of(idx, &stream);
  if (found < 0) return nullptr;
  if (found == 0) Py_RETURN_NONE;
  at::Tensor y = at::empty({B, N}, at::TensorOptions().dtype(at::kHalf).device(
                                       at::Device(at::kCUDA, (c10::DeviceIndex)idx)));
  const void* xp = x->data_ptr();
  const void* gp = g ? g->data_ptr() : nullptr;
  const void* w0p = w0->data_ptr();
  const void* w1p = w1 ? w1->data_ptr() : nullptr;
  void* yp = y.data_ptr();
  const int b = (int)B, k = (int)K, n = (int)N;
  // K split over workgroups, in a workspace that the allocator takes back in
  // stream order after this call; one launch where there is no room for it.
  at::Tensor ws;
  size_t bytes = b > 8 ? abi.gemv_workspace_bytes(g != nullptr, w1 != nullptr, b, k, n, dtype) : 0;
  if (bytes > 0) {
    try {
      ws = at::empty({(int64_t)bytes}, at::TensorOptions().dtype(at::kByte).device(y.device()));
    } catch (const c10::OutOfMemoryError&) {
      bytes = 0;
    }
  }
  void* wsp = bytes > 0 ? ws.data_ptr() : nullptr;
  int rc;
  Py_BEGIN_ALLOW_THREADS
  if (bytes > 0)
    rc = abi.gemv_ws(xp, gp, w0p, w1p, s0, s1, yp, wsp, bytes, b, k, n, (float)eps, dtype, stream);
  else if (w1)
    rc = g ? abi.f2n(xp, gp, w0p, w1p, s0, s1, yp, b, k, n, (float)eps, dtype, stream)
           : abi.f2(xp, w0p, w1p, s0, s1, yp, b, k, n, dtype, stream);
  else
    rc = g ? abi.f1(xp, gp, w0p, s0, yp, b, k, n, (float)eps, dtype, stream)
           : abi.gemv(xp, w0p, s0, yp, b, k, n, dtype, stream);
  Py_END_ALLOW_THREADS
  if (rc != DB_OK) Py_RETURN_NONE;
  return THPVariable_Wrap(dim == 1 ? y.select(0, 0) : y);
}

// (x, g, W, eps, w_scale)
PyObject* f1(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 5) Py_RETURN_NONE;
  return gemv_op(a[0], a[1], a[2], nullptr, a[3], a[4], nullptr);
  END_HANDLE_TH_ERRORS
}

// (x, W, w_scale)
PyObject* gemv(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 3) Py_RETURN_NONE;
  return gemv_op(a[0], nullptr, a[1], nullptr, nullptr, a[2], nullptr);
  END_HANDLE_TH_ERRORS
}

// (x, Wg, Wu, sg, su)
PyObject* f2(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 5) Py_RETURN_NONE;
  return gemv_op(a[0], nullptr, a[1], a[2], nullptr, a[3], a[4]);
  END_HANDLE_TH_ERRORS
}

// (x, g, Wg, Wu, eps, sg, su)
PyObject* f2n(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 7) Py_RETURN_NONE;
  return gemv_op(a[0], a[1], a[2], a[3], a[4], a[5], a[6]);
  END_HANDLE_TH_ERRORS
}

// (q, K, V, scale or None, n_splits or None): outside capture, with a
// workspace of its size already in the cache.
PyObject* f4(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 5) Py_RETURN_NONE;
  const at::Tensor *q = tensor(a[0]), *k = tensor(a[1]), *v = tensor(a[2]);
  if (!plain(q, at::kHalf, -1) || q->dim() != 3) Py_RETURN_NONE;
  const int idx = q->get_device();
  if (!plain(k, at::kHalf, idx) || !plain(v, at::kHalf, idx) || k->dim() != 4 ||
      k->sizes() != v->sizes())
    Py_RETURN_NONE;
  const int64_t B = q->size(0), Hq = q->size(1), D = q->size(2);
  const int64_t Hkv = k->size(1), L = k->size(2);
  if (k->size(0) != B || k->size(3) != D || D < 1 || B > INT_MAX || Hq > INT_MAX ||
      Hkv > INT_MAX || L > INT_MAX || D > INT_MAX)
    Py_RETURN_NONE;
  double scale = 1.0 / std::sqrt((double)D);
  if (a[3] != Py_None && !number(a[3], &scale)) Py_RETURN_NONE;
  void* stream = nullptr;
  const int found = stream_of(idx, &stream);
  if (found < 0) return nullptr;
  if (found == 0) Py_RETURN_NONE;
  PyObject* dev = PyLong_FromLong(idx);
  if (!dev) return nullptr;
  long S = 0;
  if (a[4] == Py_None) {
    PyObject* cu = PyDict_GetItemWithError(cu_counts, dev);  // borrowed
    const long cus = cu ? PyLong_AsLong(cu) : 0;
    if (cus > 0) S = abi.f4_default_splits((int)B, (int)Hkv, (int)L, (int)cus);
  } else if (PyLong_CheckExact(a[4])) {
    S = PyLong_AsLong(a[4]);
  }
  if (PyErr_Occurred() || S < 1 || S > 256) {
    PyErr_Clear();
    Py_DECREF(dev);
    Py_RETURN_NONE;
  }
  const size_t bytes =
      abi.f4_workspace_bytes((int)B, (int)Hq, (int)Hkv, (int)L, (int)D, (int)S);
  at::Tensor ws;  // keeps the workspace alive through the call
  if (bytes > 0) {
    unsigned long long capture = 0;
    if (abi.capture_id(stream, &capture) != DB_OK || capture != 0) {
      Py_DECREF(dev);
      Py_RETURN_NONE;
    }
    PyObject* key = Py_BuildValue("(OKn)", dev, (unsigned long long)(uintptr_t)stream,
                                  (Py_ssize_t)bytes);
    PyObject* hit = key ? PyDict_GetItemWithError(workspaces, key) : nullptr;  // borrowed
    Py_XDECREF(key);
    const at::Tensor* t = hit ? tensor(hit) : nullptr;
    if (!t) {
      Py_DECREF(dev);
      if (PyErr_Occurred()) return nullptr;
      Py_RETURN_NONE;
    }
    ws = *t;
  }
  Py_DECREF(dev);
  at::Tensor o = at::empty({B, Hq, D}, at::TensorOptions().dtype(at::kHalf).device(
                                           at::Device(at::kCUDA, (c10::DeviceIndex)idx)));
  const void *qp = q->data_ptr(), *kp = k->data_ptr(), *vp = v->data_ptr();
  void *op = o.data_ptr(), *wp = bytes ? ws.data_ptr() : nullptr;
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = abi.f4(qp, kp, vp, op, wp, bytes, (int)B, (int)Hq, (int)Hkv, (int)L, (int)D, (int)S,
              (float)scale, stream);
  Py_END_ALLOW_THREADS
  if (rc != DB_OK) Py_RETURN_NONE;
  return THPVariable_Wrap(o);
  END_HANDLE_TH_ERRORS
}

// (entry point addresses, raw_stream, get_device, workspaces, cu_counts)
PyObject* init(PyObject*, PyObject* args) {
  unsigned long long p[10];
  PyObject *rs, *gd, *ws, *cu;
  if (!PyArg_ParseTuple(args, "(KKKKKKKKKK)OOO!O!", &p[0], &p[1], &p[2], &p[3], &p[4], &p[5], &p[6],
                        &p[7], &p[8], &p[9], &rs, &gd, &PyDict_Type, &ws, &PyDict_Type, &cu))
    return nullptr;
  abi.f1 = reinterpret_cast<decltype(abi.f1)>((uintptr_t)p[0]);
  abi.f2 = reinterpret_cast<decltype(abi.f2)>((uintptr_t)p[1]);
  abi.f2n = reinterpret_cast<decltype(abi.f2n)>((uintptr_t)p[2]);
  abi.gemv = reinterpret_cast<decltype(abi.gemv)>((uintptr_t)p[3]);
  abi.f4_default_splits = reinterpret_cast<decltype(abi.f4_default_splits)>((uintptr_t)p[4]);
  abi.f4_workspace_bytes = reinterpret_cast<decltype(abi.f4_workspace_bytes)>((uintptr_t)p[5]);
  abi.f4 = reinterpret_cast<decltype(abi.f4)>((uintptr_t)p[6]);
  abi.capture_id = reinterpret_cast<decltype(abi.capture_id)>((uintptr_t)p[7]);
  abi.gemv_workspace_bytes = reinterpret_cast<decltype(abi.gemv_workspace_bytes)>((uintptr_t)p[8]);
  abi.gemv_ws = reinterpret_cast<decltype(abi.gemv_ws)>((uintptr_t)p[9]);
  Py_INCREF(rs);
  Py_INCREF(gd);
  Py_INCREF(ws);
  Py_INCREF(cu);
  Py_XSETREF(raw_stream, rs);
  Py_XSETREF(get_device, gd);
  Py_XSETREF(workspaces, ws);
  Py_XSETREF(cu_counts, cu);
  Py_RETURN_NONE;
}

template <PyObject* (*F)(PyObject*, PyObject* const*, Py_ssize_t)>
PyCFunction fast() {
  return reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(F));
}

PyMethodDef methods[] = {
    {"init", init, METH_VARARGS, nullptr},
    {"f1", fast<f1>(), METH_FASTCALL, nullptr},
    {"gemv", fast<gemv>(), METH_FASTCALL, nullptr},
    {"f2", fast<f2>(), METH_FASTCALL, nullptr},
    {"f2n", fast<f2n>(), METH_FASTCALL, nullptr},
    {"f4", fast<f4>(), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_fastcall", nullptr, -1, methods,
                      nullptr,               nullptr,     nullptr, nullptr};

}  // namespace

// built_for names the torch and the Python whose object layouts this module
// holds; its functions are only called where both are the running ones.
PyMODINIT_FUNC PyInit__fastcall(void) {
  PyObject* m = PyModule_Create(&module);
  if (m && PyModule_AddStringConstant(m, "built_for", DB_BUILT_FOR) < 0) Py_CLEAR(m);
  return m;
}
