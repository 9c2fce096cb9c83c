// The per-layer operators' way from Python to the C ABI (wnw_amd/_callpath.so).
//
// A decode step calls the attention once per layer; at a minute of audio the
// device needs ~10 us for it, and checking nine tensors, taking their pointers
// and converting ~20 arguments in Python took 13.7 us (now 5.1, 3.4 of them the
// launch: 30 layers of 2,586 rows 425 -> 293 us).  The functions here do
// the same for a call in its plain form: ordinary device tensors, contiguous,
// of the types and shapes the operator documents.  For any other call they
// return None and launch nothing, and the Python operator checks, copies
// or refuses as it always does, so no message or conversion is repeated here.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ops/empty.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/wnw_amd.h"

namespace {

PyObject* g_stream = nullptr;     // (device index) -> raw stream
PyObject* g_workspace = nullptr;  // (device index, stream, n_seg, group, head_dim) -> buffer tensor
PyObject* g_score_ws = nullptr;   // (device index, stream, items, heads) -> buffer tensor
PyObject* g_check = nullptr;      // (status, what): raises

// A plain tensor in device memory: no subclass, and no wrapper of a
// transform (vmap, grad levels, functionalisation) around the data.
const at::Tensor* plain(PyObject* o) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || !t.has_storage()) return nullptr;
  constexpr c10::DispatchKeySet wrapped(
      {c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::Batched,
       c10::DispatchKey::Functionalize, c10::DispatchKey::Python, c10::DispatchKey::Conjugate,
       c10::DispatchKey::Negative, c10::DispatchKey::ZeroTensor});
  if (t.key_set().has_any(wrapped)) return nullptr;
  return &t;
}
const at::Tensor* vec(PyObject* o, at::ScalarType type, int64_t n) {  // contiguous, n elements
  const at::Tensor* t = plain(o);
  return t && t->scalar_type() == type && t->numel() == n && t->is_contiguous() ? t : nullptr;
}
int dtype_code(at::ScalarType t) {
  return t == at::kFloat ? WNW_F32 : t == at::kHalf ? WNW_F16 : t == at::kBFloat16 ? WNW_BF16 : -1;
}
// [rows, d] with contiguous rows (rows > 0)
bool row_major(const at::Tensor& t, int64_t d) {
  return t.dim() == 2 && t.size(0) > 0 && t.size(1) == d && t.stride(1) == 1 && t.stride(0) == d;
}
bool number(PyObject* o, double* x) {
  if (!PyFloat_CheckExact(o) && !PyLong_CheckExact(o)) return false;
  *x = PyFloat_AsDouble(o);
  if (*x != -1.0 || !PyErr_Occurred()) return true;
  PyErr_Clear();  // beyond the type's range: the general path's to judge
  return false;
}
bool whole(PyObject* o, int64_t* x) {
  if (!PyLong_CheckExact(o)) return false;
  *x = PyLong_AsLongLong(o);
  if (*x != -1 || !PyErr_Occurred()) return true;
  PyErr_Clear();
  return false;
}

struct Ref {  // an owned reference
  PyObject* o;
  explicit Ref(PyObject* x) : o(x) {}
  ~Ref() { Py_XDECREF(o); }
  Ref(const Ref&) = delete;
  Ref& operator=(const Ref&) = delete;
};

// The current raw stream of a device, false with an exception set.
bool stream_of(int64_t index, PyObject** stream_obj, void** stream) {
  Ref idx(PyLong_FromLongLong(index));
  if (!idx.o) return false;
  *stream_obj = PyObject_CallOneArg(g_stream, idx.o);
  if (!*stream_obj) return false;
  *stream = PyLong_AsVoidPtr(*stream_obj);
  return !PyErr_Occurred();
}
const at::Tensor* buffer(const Ref& r) {
  if (!r.o) return nullptr;
  if (!THPVariable_Check(r.o)) {
    PyErr_SetString(PyExc_TypeError, "the workspace callback must return a tensor");
    return nullptr;
  }
  return &THPVariable_Unpack(r.o);
}
// Raises for a failed launch.
PyObject* failed(int rc, const char* what) {
  Ref r(PyObject_CallFunction(g_check, "is", rc, what));
  if (r.o) PyErr_SetString(PyExc_RuntimeError, what);
  return nullptr;
}

PyObject* attn_impl(PyObject* const* a) {
  const at::Tensor *q = plain(a[0]), *k = plain(a[1]), *v = plain(a[2]);
  if (!q || !k || !v || q->dim() != 3 || !q->is_contiguous()) Py_RETURN_NONE;
  const int64_t n = q->size(0), g = q->size(1), d = q->size(2);
  const int dt = dtype_code(q->scalar_type());
  if (n < 1 || dt < 0 || k->scalar_type() != q->scalar_type() || v->scalar_type() != q->scalar_type() ||
      !row_major(*k, d) || !row_major(*v, d) || k->size(0) != v->size(0))
    Py_RETURN_NONE;
  const at::Tensor* cu = vec(a[3], at::kInt, n + 1);
  double scale = 0;
  if (!cu || !number(a[4], &scale)) Py_RETURN_NONE;
  const at::Tensor* base = nullptr;
  if (a[5] != Py_None && !(base = vec(a[5], at::kLong, n))) Py_RETURN_NONE;
  int64_t rows = k->size(0);
  if (a[6] == Py_None ? base != nullptr : !whole(a[6], &rows)) Py_RETURN_NONE;
  const at::Tensor *nk = nullptr, *nv = nullptr, *cu_new = nullptr, *cap = nullptr;
  if (a[8] != Py_None) {
    if (!base || !PyTuple_CheckExact(a[8]) || PyTuple_GET_SIZE(a[8]) != 4) Py_RETURN_NONE;
    nk = vec(PyTuple_GET_ITEM(a[8], 0), q->scalar_type(), n * d);
    nv = vec(PyTuple_GET_ITEM(a[8], 1), q->scalar_type(), n * d);
    cu_new = vec(PyTuple_GET_ITEM(a[8], 2), at::kInt, n + 1);
    cap = vec(PyTuple_GET_ITEM(a[8], 3), at::kInt, n);
    if (!nk || !nv || !cu_new || !cap || nk->dim() != 2 || nv->dim() != 2 || nk->size(0) != n || nv->size(0) != n ||
        cu_new->data_ptr() == cu->data_ptr())
      Py_RETURN_NONE;
  }
  const int64_t dev = q->device().index();
  at::Tensor out;
  Ref given(nullptr);
  if (a[7] != Py_None) {
    const at::Tensor* o = plain(a[7]);
    if (!o) Py_RETURN_NONE;
    out = *o;
    given.o = Py_NewRef(a[7]);
  } else {
    out = at::empty({n, g, d}, q->options().requires_grad(false));
  }
  PyObject* so = nullptr;
  void* stream = nullptr;
  const bool has_stream = stream_of(dev, &so, &stream);
  Ref stream_ref(so);
  if (!has_stream) return nullptr;
  Ref ws(PyObject_CallFunction(g_workspace, "LOLLL", (long long)dev, so, (long long)n, (long long)g, (long long)d));
  const at::Tensor* buf = buffer(ws);
  if (!buf) return nullptr;
  void *qp = q->data_ptr(), *kp = k->data_ptr(), *vp = v->data_ptr(), *op = out.data_ptr(), *wp = buf->data_ptr();
  const int64_t wbytes = buf->numel(), kv_rows = k->size(0);
  const int32_t* cup = cu->const_data_ptr<int32_t>();
  const int64_t* bp = base ? base->const_data_ptr<int64_t>() : nullptr;
  const char* what = nk ? "decode_attn_append" : "decode_attn";
  void *nkp = nk ? nk->data_ptr() : nullptr, *nvp = nv ? nv->data_ptr() : nullptr;
  int32_t* cnp = cu_new ? cu_new->data_ptr<int32_t>() : nullptr;
  const int32_t* cpp = cap ? cap->const_data_ptr<int32_t>() : nullptr;
  int rc;
  Py_BEGIN_ALLOW_THREADS
  if (nkp)
    rc = wnw_decode_attn_append(qp, kp, vp, nkp, nvp, cup, cnp, bp, cpp, n, g, d, rows, kv_rows, (float)scale, dt, op, wp,
                                wbytes, stream);
  else
    rc = wnw_decode_attn(qp, kp, vp, cup, bp, n, g, d, rows, kv_rows, (float)scale, dt, op, wp, wbytes, stream);
  Py_END_ALLOW_THREADS
  if (rc != WNW_OK) return failed(rc, what);
  if (given.o) return Py_NewRef(given.o);
  return THPVariable_Wrap(std::move(out));
}

PyObject* score_impl(PyObject* const* a) {
  const at::Tensor *q = plain(a[0]), *k = plain(a[1]);
  if (!q || !k || q->dim() != 3 || !q->is_contiguous()) Py_RETURN_NONE;
  const int64_t n = q->size(0), h = q->size(1), d = q->size(2);
  const int dt = dtype_code(q->scalar_type());
  if (n < 1 || h < 1 || dt < 0 || k->scalar_type() != q->scalar_type() || !row_major(*k, d)) Py_RETURN_NONE;
  const at::Tensor* idx[4];
  for (int i = 0; i < 4; ++i)
    if (!(idx[i] = vec(a[2 + i], at::kInt, n))) Py_RETURN_NONE;
  const at::Tensor *acc = plain(a[6]), *off = plain(a[7]);
  if (!acc || acc->scalar_type() != at::kFloat || !acc->is_contiguous() || !off || off->scalar_type() != at::kInt ||
      !off->is_contiguous() || off->numel() < n + 1)
    Py_RETURN_NONE;
  int64_t max_audio = 0;
  if (!whole(a[8], &max_audio) || max_audio <= 0) Py_RETURN_NONE;
  double scale = 0;
  if (!number(a[9], &scale)) Py_RETURN_NONE;
  const int64_t dev = q->device().index();
  PyObject* so = nullptr;
  void* stream = nullptr;
  const bool has_stream = stream_of(dev, &so, &stream);
  Ref stream_ref(so);
  if (!has_stream) return nullptr;
  Ref ws(PyObject_CallFunction(g_score_ws, "LOLL", (long long)dev, so, (long long)n, (long long)h));
  const at::Tensor* buf = buffer(ws);
  if (!buf) return nullptr;
  void *qp = q->data_ptr(), *kp = k->data_ptr(), *wp = buf->data_ptr();
  const int32_t* ip[4];
  for (int i = 0; i < 4; ++i) ip[i] = idx[i]->const_data_ptr<int32_t>();
  float* ap = acc->data_ptr<float>();
  const int32_t* fp = off->const_data_ptr<int32_t>();
  const int64_t k_rows = k->size(0), alen = acc->numel(), wbytes = buf->numel();
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = wnw_fused_score_accumulate(qp, kp, ip[0], ip[1], ip[2], ip[3], ap, fp, n, h, d, k_rows, alen, max_audio,
                                  (float)scale, dt, wp, wbytes, stream);
  Py_END_ALLOW_THREADS
  if (rc != WNW_OK) return failed(rc, "fused_score_accumulate");
  Py_RETURN_TRUE;
}

// No C++ exception leaves an entry: such a call takes the general path.
template <PyObject* (*f)(PyObject* const*), int N>
PyObject* entry(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (n != N) {
    PyErr_Format(PyExc_TypeError, "expected %d arguments, got %zd", N, n);
    return nullptr;
  }
  if (!g_check) {
    PyErr_SetString(PyExc_RuntimeError, "setup() has not been called");
    return nullptr;
  }
  try {
    return f(args);
  } catch (const std::exception&) {
    PyErr_Clear();
    Py_RETURN_NONE;
  }
}

PyObject* setup(PyObject*, PyObject* args) {
  PyObject *s, *w, *sw, *c;
  if (!PyArg_ParseTuple(args, "OOOO", &s, &w, &sw, &c)) return nullptr;
  PyObject** dst[4] = {&g_stream, &g_workspace, &g_score_ws, &g_check};
  PyObject* src[4] = {s, w, sw, c};
  for (int i = 0; i < 4; ++i) {
    PyObject* old = *dst[i];
    *dst[i] = Py_NewRef(src[i]);
    Py_XDECREF(old);
  }
  Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"setup", setup, METH_VARARGS, "setup(raw_stream, workspace, score_workspace, check)"},
    {"attn", (PyCFunction)(void (*)(void))entry<attn_impl, 9>, METH_FASTCALL,
     "attn(q, k, v, cu, scale, seg_base, total_rows, out, append) -> out, or None: not the plain form"},
    {"score", (PyCFunction)(void (*)(void))entry<score_impl, 10>, METH_FASTCALL,
     "score(q, k, starts, ends, audio_starts, audio_ends, acc, offsets, max_audio, scale) -> True, or None: not the "
     "plain form"},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_callpath", "Plain calls of the per-layer operators.", -1, methods,
                      nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__callpath() { return PyModule_Create(&module); }
