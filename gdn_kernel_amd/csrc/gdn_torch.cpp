// CPython module gdn_kernel_amd._native: the call path of the Python entry points for the
// calls they see on every step -- plain tensors of the right dtypes and shapes, contiguous
// and on the current device.  A call that matches is launched from here; any other returns
// None, and the Python code, which has every check and message, takes it from the start.
//
// A decode of one sequence is 4.1 us on the GPU; checking ten tensors, converting nineteen
// arguments and finding the stream took 10 us a call in Python and ctypes, so that small
// calls waited for the host.
#include <Python.h>

#include <torch/csrc/autograd/python_variable.h>

#include <cstdint>
#include <initializer_list>

#include "../../include/gdn_kernel_amd.h"

namespace {

// The library's entry points (bind()).
decltype(&gdn_decode) g_decode = nullptr;
decltype(&gdn_decode_pooled) g_pooled = nullptr;
decltype(&gdn_prefill) g_prefill = nullptr;
decltype(&gdn_prefill_with_workspace) g_prefill_ws = nullptr;
PyObject* g_device = nullptr;  // torch._C._cuda_getDevice
PyObject* g_stream = nullptr;  // torch._C._cuda_getCurrentRawStream

// The tensor of a Python object: torch.Tensor or Parameter itself (no subclass, whose
// overrides the Python code would see), with memory of its own on a GPU; else null.
const at::Tensor* tensor(PyObject* o) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  return t.defined() && t.is_cuda() && t.layout() == at::kStrided && t.has_storage() ? &t : nullptr;
}

// Whether t has this dtype, device and shape and is contiguous.
bool is(const at::Tensor* t, at::ScalarType dtype, int device, std::initializer_list<int64_t> shape) {
  if (t == nullptr || t->scalar_type() != dtype || t->get_device() != device) return false;
  return t->sizes().equals(at::IntArrayRef(shape)) && t->is_contiguous();
}

// A tensor's memory, as whatever pointer an entry point takes.
struct Ptr {
  void* p;
  template <class T>
  operator T*() const {
    return static_cast<T*>(p);
  }
};
Ptr ptr(const at::Tensor* t) { return Ptr{t == nullptr || t->numel() == 0 ? nullptr : t->data_ptr()}; }

// The scale argument: None (0, the default scale) or a number that is plainly a double.
bool scale_of(PyObject* o, double* scale) {
  if (o == Py_None) {
    *scale = 0.0;
    return true;
  }
  if (!PyFloat_CheckExact(o)) return false;
  *scale = PyFloat_AS_DOUBLE(o);
  return true;
}

// The current stream of `device`, which has to be the current device.
bool stream_of(int device, void** stream) {
  PyObject* d = PyObject_CallNoArgs(g_device);
  const long current = d ? PyLong_AsLong(d) : -1;
  Py_XDECREF(d);
  if (current != device) {
    PyErr_Clear();
    return false;
  }
  PyObject* index = PyLong_FromLong(device);
  PyObject* s = index ? PyObject_CallOneArg(g_stream, index) : nullptr;
  Py_XDECREF(index);
  const unsigned long long raw = s ? PyLong_AsUnsignedLongLong(s) : 0;
  Py_XDECREF(s);
  if (PyErr_Occurred()) {
    PyErr_Clear();
    return false;
  }
  *stream = reinterpret_cast<void*>(static_cast<uintptr_t>(raw));
  return true;
}

constexpr at::ScalarType kBf16 = at::kBFloat16, kF32 = at::kFloat;

// (q, k, v, state, A_log, a, dt_bias, b, scale, output, new_state)
PyObject* decode_impl(PyObject* const* o) {
  const at::Tensor *q = tensor(o[0]), *k = tensor(o[1]), *v = tensor(o[2]), *out = tensor(o[9]), *ns = tensor(o[10]);
  if (!q || !k || !v || !out || !ns || q->dim() != 4 || k->dim() != 4 || v->dim() != 4) return nullptr;
  const int dev = q->get_device();
  const int64_t B = q->size(0), Hq = q->size(2), Hk = k->size(2), Hv = v->size(2), dk = q->size(3), dv = v->size(3);
  const at::Tensor* state = o[3] == Py_None ? nullptr : tensor(o[3]);
  const at::Tensor *A_log = tensor(o[4]), *a = tensor(o[5]), *dt = tensor(o[6]), *b = tensor(o[7]);
  double scale;
  void* stream;
  if (!is(q, kBf16, dev, {B, 1, Hq, dk}) || !is(k, kBf16, dev, {B, 1, Hk, dk}) || !is(v, kBf16, dev, {B, 1, Hv, dv}) ||
      (o[3] != Py_None && !is(state, kF32, dev, {B, Hv, dv, dk})) || !is(A_log, kF32, dev, {Hv}) ||
      !is(a, kBf16, dev, {B, 1, Hv}) || !is(dt, kF32, dev, {Hv}) || !is(b, kBf16, dev, {B, 1, Hv}) ||
      !is(out, kBf16, dev, {B, 1, Hv, dv}) || !is(ns, kF32, dev, {B, Hv, dv, dk}) || !scale_of(o[8], &scale) ||
      Hq > INT32_MAX || Hk > INT32_MAX || Hv > INT32_MAX || dk > INT32_MAX || dv > INT32_MAX || !stream_of(dev, &stream))
    return nullptr;
  const Ptr pq = ptr(q), pk = ptr(k), pv = ptr(v), ps = ptr(state), pA = ptr(A_log), pa = ptr(a), pd = ptr(dt),
            pb = ptr(b), po = ptr(out), pn = ptr(ns);
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = g_decode(pq, pk, pv, ps, pA, pa, pd, pb, scale, po, pn, B, int32_t(Hq), int32_t(Hk), int32_t(Hv), int32_t(dk),
                int32_t(dv), stream);
  Py_END_ALLOW_THREADS
  return PyLong_FromLong(rc);
}

// (q, k, v, state_pool, A_log, a, dt_bias, b, scale, output, state_indices)
PyObject* pooled_impl(PyObject* const* o) {
  const at::Tensor *q = tensor(o[0]), *k = tensor(o[1]), *v = tensor(o[2]), *pool = tensor(o[3]), *out = tensor(o[9]),
                   *idx = tensor(o[10]);
  if (!q || !k || !v || !pool || !out || !idx || q->dim() != 4 || k->dim() != 4 || v->dim() != 4 || pool->dim() != 4)
    return nullptr;
  const int dev = q->get_device();
  const int64_t B = q->size(0), Hq = q->size(2), Hk = k->size(2), Hv = v->size(2), dk = q->size(3), dv = v->size(3);
  const int64_t slots = pool->size(0);
  const at::Tensor *A_log = tensor(o[4]), *a = tensor(o[5]), *dt = tensor(o[6]), *b = tensor(o[7]);
  double scale;
  void* stream;
  if (!is(q, kBf16, dev, {B, 1, Hq, dk}) || !is(k, kBf16, dev, {B, 1, Hk, dk}) || !is(v, kBf16, dev, {B, 1, Hv, dv}) ||
      !is(pool, kF32, dev, {slots, Hv, dv, dk}) || !is(idx, at::kInt, dev, {B}) || !is(A_log, kF32, dev, {Hv}) ||
      !is(a, kBf16, dev, {B, 1, Hv}) || !is(dt, kF32, dev, {Hv}) || !is(b, kBf16, dev, {B, 1, Hv}) ||
      !is(out, kBf16, dev, {B, 1, Hv, dv}) || !scale_of(o[8], &scale) || Hq > INT32_MAX || Hk > INT32_MAX ||
      Hv > INT32_MAX || dk > INT32_MAX || dv > INT32_MAX || !stream_of(dev, &stream))
    return nullptr;
  const Ptr pq = ptr(q), pk = ptr(k), pv = ptr(v), pi = ptr(idx), pA = ptr(A_log), pa = ptr(a), pd = ptr(dt),
            pb = ptr(b), pp = ptr(pool), po = ptr(out);
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = g_pooled(pq, pk, pv, pp, slots, pi, pA, pa, pd, pb, scale, po, B, int32_t(Hq), int32_t(Hk), int32_t(Hv),
                int32_t(dk), int32_t(dv), stream);
  Py_END_ALLOW_THREADS
  return PyLong_FromLong(rc);
}

// (q, k, v, state, A_log, a, dt_bias, b, cu_seqlens, scale, output, new_state[, workspace])
PyObject* prefill_impl(PyObject* const* o, bool with_workspace) {
  const at::Tensor *q = tensor(o[0]), *k = tensor(o[1]), *v = tensor(o[2]), *cu = tensor(o[8]), *out = tensor(o[10]),
                   *ns = tensor(o[11]);
  if (!q || !k || !v || !cu || !out || !ns || q->dim() != 3 || k->dim() != 3 || v->dim() != 3 || cu->dim() != 1 ||
      cu->size(0) < 1)
    return nullptr;
  const int dev = q->get_device();
  const int64_t T = q->size(0), Hq = q->size(1), Hk = k->size(1), Hv = v->size(1), dk = q->size(2), dv = v->size(2);
  const int64_t N = cu->size(0) - 1;
  const bool cu64 = cu->scalar_type() == at::kLong;
  const at::Tensor* state = o[3] == Py_None ? nullptr : tensor(o[3]);
  const at::Tensor *A_log = tensor(o[4]), *a = tensor(o[5]), *dt = tensor(o[6]), *b = tensor(o[7]);
  const at::Tensor* ws = nullptr;
  if (with_workspace && o[12] != Py_None) {
    ws = tensor(o[12]);
    if (!ws || ws->dim() != 1 || !is(ws, at::kByte, dev, {ws->size(0)})) return nullptr;
  }
  double scale;
  void* stream;
  if (!is(cu, cu64 ? at::kLong : at::kInt, dev, {N + 1}) || !is(q, kBf16, dev, {T, Hq, dk}) ||
      !is(k, kBf16, dev, {T, Hk, dk}) || !is(v, kBf16, dev, {T, Hv, dv}) ||
      (o[3] != Py_None && !is(state, kF32, dev, {N, Hv, dv, dk})) || !is(A_log, kF32, dev, {Hv}) ||
      !is(a, kBf16, dev, {T, Hv}) || !is(dt, kF32, dev, {Hv}) || !is(b, kBf16, dev, {T, Hv}) ||
      !is(out, kBf16, dev, {T, Hv, dv}) || !is(ns, kF32, dev, {N, Hv, dv, dk}) || !scale_of(o[9], &scale) ||
      Hq > INT32_MAX || Hk > INT32_MAX || Hv > INT32_MAX || dk > INT32_MAX || dv > INT32_MAX || !stream_of(dev, &stream))
    return nullptr;
  const Ptr pq = ptr(q), pk = ptr(k), pv = ptr(v), ps = ptr(state), pA = ptr(A_log), pa = ptr(a), pd = ptr(dt),
            pb = ptr(b), pc = Ptr{cu->data_ptr()}, po = ptr(out), pn = ptr(ns), pw = ptr(ws);
  const int64_t wn = ws ? ws->size(0) : 0;
  int rc;
  Py_BEGIN_ALLOW_THREADS
  if (with_workspace) {
    rc = g_prefill_ws(pq, pk, pv, ps, pA, pa, pd, pb, pc, cu64, N, T, scale, po, pn, int32_t(Hq), int32_t(Hk),
                      int32_t(Hv), int32_t(dk), int32_t(dv), pw, wn, stream);
  } else {
    rc = g_prefill(pq, pk, pv, ps, pA, pa, pd, pb, pc, cu64, N, T, scale, po, pn, int32_t(Hq), int32_t(Hk), int32_t(Hv),
                   int32_t(dk), int32_t(dv), stream);
  }
  Py_END_ALLOW_THREADS
  return PyLong_FromLong(rc);
}

// Runs `f`; None where it launched nothing (a C++ exception included: the Python code
// meets the same condition and reports it).
template <class F>
PyObject* or_none(Py_ssize_t n, Py_ssize_t want, F&& f) {
  if (n != want) {
    PyErr_Format(PyExc_TypeError, "expected %zd arguments (got %zd)", want, n);
    return nullptr;
  }
  PyObject* r = nullptr;
  try {
    r = f();
  } catch (...) {
    r = nullptr;
  }
  if (r == nullptr && !PyErr_Occurred()) Py_RETURN_NONE;
  return r;
}

PyObject* py_decode(PyObject*, PyObject* const* o, Py_ssize_t n) {
  return or_none(n, 11, [&] { return decode_impl(o); });
}
PyObject* py_pooled(PyObject*, PyObject* const* o, Py_ssize_t n) {
  return or_none(n, 11, [&] { return pooled_impl(o); });
}
PyObject* py_prefill(PyObject*, PyObject* const* o, Py_ssize_t n) {
  return or_none(n, 12, [&] { return prefill_impl(o, false); });
}
PyObject* py_prefill_ws(PyObject*, PyObject* const* o, Py_ssize_t n) {
  return or_none(n, 13, [&] { return prefill_impl(o, true); });
}

// bind(decode, decode_pooled, prefill, prefill_with_workspace, device, stream): the
// addresses of the library's entry points, and torch's current-device and raw-stream
// functions.
PyObject* py_bind(PyObject*, PyObject* args) {
  unsigned long long d, dp, pf, pw;
  PyObject *device, *stream;
  if (!PyArg_ParseTuple(args, "KKKKOO", &d, &dp, &pf, &pw, &device, &stream)) return nullptr;
  g_decode = reinterpret_cast<decltype(g_decode)>(static_cast<uintptr_t>(d));
  g_pooled = reinterpret_cast<decltype(g_pooled)>(static_cast<uintptr_t>(dp));
  g_prefill = reinterpret_cast<decltype(g_prefill)>(static_cast<uintptr_t>(pf));
  g_prefill_ws = reinterpret_cast<decltype(g_prefill_ws)>(static_cast<uintptr_t>(pw));
  Py_INCREF(device);
  Py_INCREF(stream);
  Py_XSETREF(g_device, device);
  Py_XSETREF(g_stream, stream);
  Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"bind", py_bind, METH_VARARGS, nullptr},
    {"decode", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(py_decode)), METH_FASTCALL, nullptr},
    {"decode_pooled", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(py_pooled)), METH_FASTCALL, nullptr},
    {"prefill", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(py_prefill)), METH_FASTCALL, nullptr},
    {"prefill_with_workspace", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(py_prefill_ws)),
     METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_native", "Call path of the gdn_kernel_amd entry points.", -1, methods,
                      nullptr, nullptr, nullptr, nullptr};

}  // namespace

// The module is compiled against one torch (it reads tensors in place) and one library (it
// calls the addresses it is given); the loader compares all three stamps.
#ifndef GDN_NATIVE_TORCH
#define GDN_NATIVE_TORCH "unknown"
#define GDN_NATIVE_LIBRARY "unknown"
#define GDN_NATIVE_BUILD_ID "unknown"
#endif
PyMODINIT_FUNC PyInit__native(void) {
  PyObject* m = PyModule_Create(&module);
  if (m == nullptr) return nullptr;
  if (PyModule_AddStringConstant(m, "torch_version", GDN_NATIVE_TORCH) != 0 ||
      PyModule_AddStringConstant(m, "library_build_id", GDN_NATIVE_LIBRARY) != 0 ||
      PyModule_AddStringConstant(m, "build_id", GDN_NATIVE_BUILD_ID) != 0) {
    Py_DECREF(m);
    return nullptr;
  }
  return m;
}
