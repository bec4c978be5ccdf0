// rq_bind.cpp -- the Python calls of one layer on librq without ctypes.
//
// runtimed_amd/rq.py calls librq through ctypes: about 10 us of host time a
// call (the output's torch.empty, the current stream's Python object, a
// conversion an argument), more than most decode kernels run.  These functions
// do the same work for the plain form of a call -- contiguous tensors of a
// supported type on a GPU, no subclass and no transform around them -- and
// return the outputs, a negative rq_status (the caller raises it), or None
// where the call is not of that form (the caller then takes its general path).
// Outputs come from the caching allocator on the current stream and the GIL is
// released around librq, as in the general path.
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/rq.h"

namespace {

PyObject *g_hv, *g_n;  // interned attribute names of a weight

// The library's code of a scalar type, or -1.
int ftype(at::ScalarType t) {
  switch (t) {
    case at::kFloat: return RQ_F32;
    case at::kHalf: return RQ_F16;
    case at::kBFloat16: return RQ_BF16;
    default: return -1;
  }
}

// A tensor whose memory may be handed to the library: dense, on a GPU, no
// Python subclass, not a functorch or functionalization wrapper.
const at::Tensor *plain(PyObject *o) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor &t = THPVariable_Unpack(o);
  if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || !t.has_storage()) return nullptr;
  const c10::DispatchKeySet ks = t.key_set();
  if (ks.has(c10::DispatchKey::FuncTorchBatched) || ks.has(c10::DispatchKey::FuncTorchGradWrapper) ||
      ks.has(c10::DispatchKey::Functionalize) || ks.has(c10::DispatchKey::Python) || !t.is_contiguous())
    return nullptr;
  return &t;
}

void *stream_of(const at::Tensor &t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

at::Tensor empty_as(const at::Tensor &x, at::IntArrayRef shape, at::ScalarType dt) {
  return at::empty(shape, x.options().dtype(dt).requires_grad(false));
}

// Output type: a torch.dtype, or None for the input's.  false: not a type the
// library writes.
bool out_type(PyObject *o, const at::Tensor &x, at::ScalarType *dt) {
  if (o == Py_None) *dt = x.scalar_type();
  else if (THPDtype_Check(o)) *dt = reinterpret_cast<THPDtype *>(o)->scalar_type;
  else return false;
  return ftype(*dt) >= 0;
}

#define RQ_CALL(rc, call)       \
  int rc;                       \
  Py_BEGIN_ALLOW_THREADS        \
  rc = (call);                  \
  Py_END_ALLOW_THREADS          \
  if (rc != 0) return PyLong_FromLong(rc)

// linear(weight, x, out_dtype or None, bias or None)
PyObject *b_linear(PyObject *, PyObject *const *a, Py_ssize_t na) {
  HANDLE_TH_ERRORS
  if (na != 4) Py_RETURN_NONE;
  const at::Tensor *x = plain(a[1]), *bias = nullptr;
  at::ScalarType dt;
  if (!x || x->dim() < 1 || ftype(x->scalar_type()) < 0 || !out_type(a[2], *x, &dt)) Py_RETURN_NONE;
  if (a[3] != Py_None) {
    bias = plain(a[3]);
    if (!bias || ftype(bias->scalar_type()) < 0) Py_RETURN_NONE;
  }
  long n = 0;
  const rq_weight *h = nullptr;
  {
    PyObject *o = PyObject_GetAttr(a[0], g_n), *p = o ? PyObject_GetAttr(a[0], g_hv) : nullptr;
    if (p) n = PyLong_AsLong(o), h = static_cast<const rq_weight *>(PyLong_AsVoidPtr(p));
    Py_XDECREF(o);
    Py_XDECREF(p);
    if (PyErr_Occurred()) return nullptr;
  }
  const int64_t k = x->size(-1), rows = k ? x->numel() / k : 0;
  at::DimVector shape(x->sizes());
  shape.back() = n;
  at::Tensor y = empty_as(*x, shape, dt);
  RQ_CALL(rc, rq_linear_bias(h, x->data_ptr(), ftype(x->scalar_type()), rows, k, bias ? bias->data_ptr() : nullptr,
                             bias ? ftype(bias->scalar_type()) : RQ_F32, y.data_ptr(), ftype(dt), stream_of(*x)));
  return THPVariable_Wrap(std::move(y));
  END_HANDLE_TH_ERRORS
}

// linear_multi(weights, x, biases or None, out_dtype or None) -> list
PyObject *b_linear_multi(PyObject *, PyObject *const *a, Py_ssize_t na) {
  HANDLE_TH_ERRORS
  constexpr int kMax = 8;
  if (na != 4 || !(PyList_CheckExact(a[0]) || PyTuple_CheckExact(a[0]))) Py_RETURN_NONE;
  const Py_ssize_t count = PySequence_Fast_GET_SIZE(a[0]);
  const at::Tensor *x = plain(a[1]);
  at::ScalarType dt;
  if (count < 1 || count > kMax || !x || x->dim() < 1 || ftype(x->scalar_type()) < 0 || !out_type(a[3], *x, &dt))
    Py_RETURN_NONE;
  const void *bs[kMax] = {};
  at::ScalarType bt = at::kFloat;
  if (a[2] != Py_None) {
    if (!(PyList_CheckExact(a[2]) || PyTuple_CheckExact(a[2])) || PySequence_Fast_GET_SIZE(a[2]) != count)
      Py_RETURN_NONE;
    bool first = true;
    for (Py_ssize_t i = 0; i < count; ++i) {
      PyObject *o = PySequence_Fast_GET_ITEM(a[2], i);
      if (o == Py_None) continue;
      const at::Tensor *b = plain(o);
      if (!b || ftype(b->scalar_type()) < 0 || (!first && b->scalar_type() != bt)) Py_RETURN_NONE;
      bt = b->scalar_type();
      first = false;
      bs[i] = b->data_ptr();
    }
  }
  const rq_weight *hs[kMax];
  void *ys[kMax];
  at::Tensor out[kMax];
  const int64_t k = x->size(-1), rows = k ? x->numel() / k : 0;
  at::DimVector shape(x->sizes());
  for (Py_ssize_t i = 0; i < count; ++i) {
    PyObject *w = PySequence_Fast_GET_ITEM(a[0], i);
    PyObject *o = PyObject_GetAttr(w, g_n), *p = o ? PyObject_GetAttr(w, g_hv) : nullptr;
    if (p) shape.back() = PyLong_AsLong(o), hs[i] = static_cast<const rq_weight *>(PyLong_AsVoidPtr(p));
    Py_XDECREF(o);
    Py_XDECREF(p);
    if (PyErr_Occurred()) return nullptr;
    out[i] = empty_as(*x, shape, dt);
    ys[i] = out[i].data_ptr();
  }
  RQ_CALL(rc, rq_linear_multi((int)count, hs, x->data_ptr(), ftype(x->scalar_type()), rows, k,
                              a[2] != Py_None ? bs : nullptr, ftype(bt), ys, ftype(dt), stream_of(*x)));
  PyObject *list = PyList_New(count);
  if (!list) return nullptr;
  for (Py_ssize_t i = 0; i < count; ++i) {
    PyObject *t = THPVariable_Wrap(std::move(out[i]));
    if (!t) {
      Py_DECREF(list);
      return nullptr;
    }
    PyList_SET_ITEM(list, i, t);
  }
  return list;
  END_HANDLE_TH_ERRORS
}

// fp8_gemm(x, w, w_scale or None, mode, out_dtype)
PyObject *b_fp8_gemm(PyObject *, PyObject *const *a, Py_ssize_t na) {
  HANDLE_TH_ERRORS
  if (na != 5) Py_RETURN_NONE;
  const at::Tensor *x = plain(a[0]), *w = plain(a[1]), *ws = nullptr;
  at::ScalarType dt;
  if (!x || !w || x->dim() < 1 || w->dim() != 2 || ftype(x->scalar_type()) < 0 || w->element_size() != 1 ||
      a[4] == Py_None || !out_type(a[4], *x, &dt) || x->size(-1) != w->size(1) || w->size(1) == 0)
    Py_RETURN_NONE;
  if (a[2] != Py_None) {
    ws = plain(a[2]);
    if (!ws || ws->scalar_type() != at::kFloat) Py_RETURN_NONE;
  }
  const long mode = PyLong_AsLong(a[3]);
  if (mode == -1 && PyErr_Occurred()) return nullptr;
  const int64_t n = w->size(0), k = w->size(1), m = x->numel() / k;
  at::DimVector shape(x->sizes());
  shape.back() = n;
  at::Tensor y = empty_as(*x, shape, dt);
  RQ_CALL(rc, rq_fp8_gemm(x->data_ptr(), ftype(x->scalar_type()), m, static_cast<const uint8_t *>(w->data_ptr()),
                          ws ? static_cast<const float *>(ws->data_ptr()) : nullptr, n, k, y.data_ptr(), ftype(dt),
                          (int)mode, stream_of(*x)));
  return THPVariable_Wrap(std::move(y));
  END_HANDLE_TH_ERRORS
}

// marlin(x, packed, scales, in_dim, out_dim)
PyObject *b_marlin(PyObject *, PyObject *const *a, Py_ssize_t na) {
  HANDLE_TH_ERRORS
  if (na != 5) Py_RETURN_NONE;
  const at::Tensor *x = plain(a[0]), *w = plain(a[1]), *s = plain(a[2]);
  const long k = PyLong_AsLong(a[3]), n = PyLong_AsLong(a[4]);
  if (PyErr_Occurred()) return nullptr;
  if (!x || !w || !s || x->dim() < 1 || ftype(x->scalar_type()) < 0 || s->scalar_type() != at::kFloat || k < 1 ||
      n < 1 || x->size(-1) != k || x->numel() == 0)
    Py_RETURN_NONE;
  at::DimVector shape(x->sizes());
  shape.back() = n;
  at::Tensor y = empty_as(*x, shape, x->scalar_type());
  const int xt = ftype(x->scalar_type());
  RQ_CALL(rc, rq_marlin_linear(static_cast<const uint32_t *>(w->data_ptr()), static_cast<const float *>(s->data_ptr()),
                               n, k, x->data_ptr(), xt, x->numel() / k, y.data_ptr(), xt, stream_of(*x)));
  return THPVariable_Wrap(std::move(y));
  END_HANDLE_TH_ERRORS
}

// kv_pair(k, v, mode, code dtype) -> (kq, k scales, vq, v scales)
PyObject *b_kv_pair(PyObject *, PyObject *const *a, Py_ssize_t na) {
  HANDLE_TH_ERRORS
  if (na != 4 || !THPDtype_Check(a[3])) Py_RETURN_NONE;
  const at::Tensor *k = plain(a[0]), *v = plain(a[1]);
  if (!k || !v || k->dim() != 4 || k->sizes() != v->sizes() || k->scalar_type() != v->scalar_type() ||
      k->device() != v->device() || ftype(k->scalar_type()) < 0)
    Py_RETURN_NONE;
  const long mode = PyLong_AsLong(a[2]);
  if (mode == -1 && PyErr_Occurred()) return nullptr;
  const at::ScalarType qt = reinterpret_cast<THPDtype *>(a[3])->scalar_type;
  const int64_t h = k->size(1);
  at::Tensor out[4] = {empty_as(*k, k->sizes(), qt), empty_as(*k, {1, h, 1, 1}, at::kFloat),
                       empty_as(*k, k->sizes(), qt), empty_as(*k, {1, h, 1, 1}, at::kFloat)};
  RQ_CALL(rc, rq_kv_quantize_pair(k->data_ptr(), v->data_ptr(), ftype(k->scalar_type()), k->size(0), h,
                                  k->size(2) * k->size(3), (int)mode, out[0].data_ptr(), out[2].data_ptr(),
                                  static_cast<float *>(out[1].data_ptr()), static_cast<float *>(out[3].data_ptr()),
                                  stream_of(*k)));
  PyObject *r[4];
  for (int i = 0; i < 4; ++i) r[i] = THPVariable_Wrap(std::move(out[i]));
  PyObject *t = r[0] && r[1] && r[2] && r[3] ? PyTuple_Pack(4, r[0], r[1], r[2], r[3]) : nullptr;
  for (PyObject *o : r) Py_XDECREF(o);
  return t;
  END_HANDLE_TH_ERRORS
}

// kv_dequantize(q, scale, mode, target dtype)
PyObject *b_kv_dequantize(PyObject *, PyObject *const *a, Py_ssize_t na) {
  HANDLE_TH_ERRORS
  if (na != 4 || !THPDtype_Check(a[3])) Py_RETURN_NONE;
  const at::Tensor *q = plain(a[0]), *s = plain(a[1]);
  const at::ScalarType dt = reinterpret_cast<THPDtype *>(a[3])->scalar_type;
  const long mode = PyLong_AsLong(a[2]);
  if (mode == -1 && PyErr_Occurred()) return nullptr;
  if (!q || !s || q->dim() != 4 || q->element_size() != (mode == RQ_KV_F16 ? 2 : 1) || s->scalar_type() != at::kFloat ||
      s->numel() != q->size(1) || ftype(dt) < 0)
    Py_RETURN_NONE;
  at::Tensor y = empty_as(*q, q->sizes(), dt);
  RQ_CALL(rc, rq_kv_dequantize(q->data_ptr(), (int)mode, static_cast<const float *>(s->data_ptr()), q->size(0),
                               q->size(1), q->size(2) * q->size(3), y.data_ptr(), ftype(dt), stream_of(*q)));
  return THPVariable_Wrap(std::move(y));
  END_HANDLE_TH_ERRORS
}

// dequantize(weight handle, n, k, device index)
PyObject *b_dequantize(PyObject *, PyObject *const *a, Py_ssize_t na) {
  HANDLE_TH_ERRORS
  if (na != 4) Py_RETURN_NONE;
  const void *h = PyLong_AsVoidPtr(a[0]);
  const long n = PyLong_AsLong(a[1]), k = PyLong_AsLong(a[2]), dev = PyLong_AsLong(a[3]);
  if (PyErr_Occurred()) return nullptr;
  at::Tensor y = at::empty({n, k}, at::TensorOptions().dtype(at::kFloat).device(at::kCUDA, (c10::DeviceIndex)dev));
  RQ_CALL(rc, rq_dequant_f32(static_cast<const rq_weight *>(h), static_cast<float *>(y.data_ptr()), stream_of(y)));
  return THPVariable_Wrap(std::move(y));
  END_HANDLE_TH_ERRORS
}

// embedding(weight handle, k, device index, u32 ids as a buffer)
PyObject *b_embedding(PyObject *, PyObject *const *a, Py_ssize_t na) {
  HANDLE_TH_ERRORS
  if (na != 4) Py_RETURN_NONE;
  const void *h = PyLong_AsVoidPtr(a[0]);
  const long k = PyLong_AsLong(a[1]), dev = PyLong_AsLong(a[2]);
  Py_buffer buf;
  if (PyErr_Occurred() || PyObject_GetBuffer(a[3], &buf, PyBUF_C_CONTIGUOUS) != 0) return nullptr;
  at::Tensor y;
  int rc = 0;
  try {
    y = at::empty({buf.len / 4, k}, at::TensorOptions().dtype(at::kFloat).device(at::kCUDA, (c10::DeviceIndex)dev));
    void *s = stream_of(y);
    Py_BEGIN_ALLOW_THREADS
    rc = rq_embedding(static_cast<const rq_weight *>(h), static_cast<const uint32_t *>(buf.buf), buf.len / 4,
                      static_cast<float *>(y.data_ptr()), s);
    Py_END_ALLOW_THREADS
  } catch (...) {
    PyBuffer_Release(&buf);
    throw;
  }
  PyBuffer_Release(&buf);
  if (rc != 0) return PyLong_FromLong(rc);
  return THPVariable_Wrap(std::move(y));
  END_HANDLE_TH_ERRORS
}

#define RQ_DEF(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(b_##name)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {RQ_DEF(linear),  RQ_DEF(linear_multi),  RQ_DEF(fp8_gemm),  RQ_DEF(marlin),
                         RQ_DEF(kv_pair), RQ_DEF(kv_dequantize), RQ_DEF(embedding),
                         RQ_DEF(dequantize), {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_rqc", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__rqc() {
  g_hv = PyUnicode_InternFromString("_hv");
  g_n = PyUnicode_InternFromString("n");
  return g_hv && g_n ? PyModule_Create(&module) : nullptr;
}
