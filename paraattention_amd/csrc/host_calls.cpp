// The host side of the ops' ordinary calls in native code: operand checks, output and workspace allocation and the call into
// libparaattn_hip.so.  In Python these took 15 us of an attention call whose kernel takes 10 (and 5 us of a launch);
// here they take 5.  Every function returns None for a call that is not of the ordinary kind -- operands on several
// devices, of other types or shapes, rows that need a copy first -- and the Python code in ops.py decides what becomes of it; an
// integer is the library's error code.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <torch/csrc/Exceptions.h>
#include <dlfcn.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cmath>
#include <vector>

#include "../../include/paraattn_hip.h"

namespace {

using at::Tensor;

// The entries of the library that _lib.py has loaded, looked up in that very one (another build of it may be in use).
#define ENTRIES(X) \
  X(pa_attn_fwd_blocksparse) \
  X(pa_attn_fwd_call_workspace_bytes) \
  X(pa_attn_fwd_lse_ws) \
  X(pa_attn_fwd_masked) \
  X(pa_attn_fwd_masked_call_workspace_bytes) \
  X(pa_attn_fwd_narrow) \
  X(pa_attn_fwd_narrow_plan) \
  X(pa_blocksparse_workspace_bytes) \
  X(pa_fbcache_apply_residual) \
  X(pa_fbcache_apply_residual2) \
  X(pa_fbcache_residual) \
  X(pa_fbcache_residual_ratio) \
  X(pa_fbcache_residual_ratio_strided) \
  X(pa_taylorseer_update) \
  X(pa_taylorseer_value)
struct Library {
#define MEMBER(name) decltype(&::name) name;
  ENTRIES(MEMBER)
#undef MEMBER
};
Library lib = {};

// bind(handle of the loaded library): before any other function of this module
PyObject* bind(PyObject*, PyObject* arg) {
  void* const handle = PyLong_AsVoidPtr(arg);
  if (PyErr_Occurred()) return nullptr;
#define LOOK_UP(entry)                                                                                                  \
  if ((lib.entry = (decltype(&::entry))dlsym(handle, #entry)) == nullptr) {                                             \
    PyErr_SetString(PyExc_ImportError, #entry " is missing in the loaded library");                                     \
    return nullptr;                                                                                                     \
  }
  ENTRIES(LOOK_UP)
#undef LOOK_UP
  Py_RETURN_NONE;
}

// The C++ handle of a tensor, null for None; false (and no error set): neither
bool optional_tensor(PyObject* o, const Tensor** out) {
  *out = nullptr;
  if (o == Py_None) return true;
  if (!THPVariable_Check(o)) return false;
  *out = &THPVariable_Unpack(o);
  return true;
}

int dtype_code(at::ScalarType t) {
  switch (t) {
    case at::kBFloat16: return PA_DTYPE_BF16;
    case at::kHalf: return PA_DTYPE_F16;
    case at::kFloat: return PA_DTYPE_F32;
    default: return -1;
  }
}

// unit-stride rows whose starts are 16-byte aligned, as the kernels' vector loads need them
bool vector_rows(const Tensor& t) {
  const auto st = t.strides(), sz = t.sizes();
  const size_t n = st.size();
  if (n == 0 || st[n - 1] != 1) return false;
  for (size_t i = 0; i + 1 < n; ++i)
    if (st[i] % 8 != 0 && sz[i] > 1) return false;
  return true;
}
bool kernel_ready(const Tensor& t) { return vector_rows(t) && (uintptr_t)t.data_ptr() % 16 == 0; }

struct Strides3 {
  int64_t v[3];
  explicit Strides3(const Tensor& t) {
    for (int i = 0; i < 3; ++i) v[i] = t.size(i) == 1 ? 0 : t.stride(i);
  }
};

Tensor out_like(const Tensor& q) {  // the query's own memory layout where the kernels can write it
  Tensor out = at::empty_like(q);
  return vector_rows(out) ? out : at::empty(q.sizes(), q.options());
}
Tensor scratch(size_t bytes, const Tensor& like) { return bytes ? at::empty({(int64_t)bytes}, like.options().dtype(at::kByte)) : Tensor(); }
void* ptr(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }

bool plain(const Tensor& t) { return t.layout() == at::kStrided && t.is_cuda() && !t.is_conj() && !t.is_neg(); }

PyObject* pair(const Tensor& a, const Tensor& b) {
  PyObject* r = PyTuple_New(2);
  if (!r) return nullptr;
  PyTuple_SET_ITEM(r, 0, THPVariable_Wrap(a));
  if (b.defined()) PyTuple_SET_ITEM(r, 1, THPVariable_Wrap(b));
  else {
    Py_INCREF(Py_None);
    PyTuple_SET_ITEM(r, 1, Py_None);
  }
  return r;
}

// query, key and value as the attention kernels take them without a copy
bool attention_operands(const Tensor& q, const Tensor& k, const Tensor& v) {
  if (q.dim() != 4 || k.dim() != 4 || v.dim() != 4 || !plain(q) || !plain(k) || !plain(v)) return false;
  if (q.scalar_type() != at::kBFloat16 && q.scalar_type() != at::kHalf) return false;
  if (k.scalar_type() != q.scalar_type() || v.scalar_type() != q.scalar_type()) return false;
  if (k.device() != q.device() || v.device() != q.device()) return false;
  if (k.size(0) != q.size(0) || k.size(1) != q.size(1) || k.size(3) != q.size(3) || v.sizes() != k.sizes()) return false;
  return q.numel() > 0 && k.numel() > 0 && kernel_ready(q) && kernel_ready(k) && kernel_ready(v);
}

// attention(query, key, value, attn_mask or None, scale or None, want_lse, is_causal, stream) -> (out, lse or None)
PyObject* attention(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  const Tensor *pq, *pk, *pv, *pm;
  if (nargs != 8 || !optional_tensor(args[0], &pq) || !optional_tensor(args[1], &pk) || !optional_tensor(args[2], &pv) || !optional_tensor(args[3], &pm))
    Py_RETURN_NONE;
  if (!pq || !pk || !pv || !attention_operands(*pq, *pk, *pv)) Py_RETURN_NONE;
  const Tensor &q = *pq, &k = *pk, &v = *pv;
  const int64_t B = q.size(0), H = q.size(1), Sq = q.size(2), D = q.size(3), Skv = k.size(2);
  if (B > INT32_MAX || H > INT32_MAX || Sq > INT32_MAX || Skv > INT32_MAX) Py_RETURN_NONE;
  const bool native = D == 64 || D == 128;
  if (!native && (pm != nullptr || D % 8 != 0 || D > 96)) Py_RETURN_NONE;
  const int causal = PyObject_IsTrue(args[6]);
  if (causal && pm != nullptr) Py_RETURN_NONE;
  double scale = 1.0 / std::sqrt((double)D);
  if (args[4] != Py_None) {
    scale = PyFloat_AsDouble(args[4]);
    if (PyErr_Occurred()) return nullptr;
  }
  const bool want_lse = PyObject_IsTrue(args[5]);
  void* const stream = PyLong_AsVoidPtr(args[7]);
  if (PyErr_Occurred()) return nullptr;
  int kind = 0;
  int64_t ms[4] = {0, 0, 0, 0};
  if (pm != nullptr) {
    const Tensor& m = *pm;
    if (!plain(m) || m.device() != q.device() || m.dim() > 4) Py_RETURN_NONE;
    kind = m.scalar_type() == at::kBool ? PA_MASK_BOOL : m.scalar_type() == at::kFloat ? PA_MASK_F32 : m.scalar_type() == q.scalar_type() ? PA_MASK_ACT : 0;
    if (kind == 0) Py_RETURN_NONE;
    const int64_t full[4] = {B, H, Sq, Skv};
    for (int64_t d = 0, lead = 4 - m.dim(); d < m.dim(); ++d) {
      const int64_t n = m.size(d);
      if (n != 1 && n != full[lead + d]) Py_RETURN_NONE;
      ms[lead + d] = n == 1 ? 0 : m.stride(d);
    }
  }
  const Strides3 qs(q), ks(k), vs(v);
  const int dt = dtype_code(q.scalar_type());
  size_t bytes = 0;
  if (pm != nullptr) bytes = lib.pa_attn_fwd_masked_call_workspace_bytes(B, H, Sq, Skv, D, ks.v, vs.v, kind, ms);
  else if (native) bytes = lib.pa_attn_fwd_call_workspace_bytes(B, H, Sq, Skv, D, ks.v, vs.v, 0, causal);
  else if (!lib.pa_attn_fwd_narrow_plan(B, H, Sq, Skv, D, ks.v, vs.v, causal, &bytes)) Py_RETURN_NONE;
  Tensor out, lse;
  int rc;
  {
    pybind11::gil_scoped_release no_gil;
    // (rows of other head_dims come out contiguous, as from the zero-padded copies)
    out = native ? out_like(q) : at::empty(q.sizes(), q.options());
    if (want_lse) lse = at::empty({B, H, Sq}, q.options().dtype(at::kFloat));
    const Tensor ws = scratch(bytes, q);
    const Strides3 os(out);
    if (pm != nullptr)
      rc = lib.pa_attn_fwd_masked(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), (float*)ptr(lse), dt, B, H, Sq, Skv, D, qs.v, ks.v, vs.v, os.v,
                              (float)scale, pm->data_ptr(), kind, ms, ptr(ws), bytes, stream);
    else if (native)
      rc = lib.pa_attn_fwd_lse_ws(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), (float*)ptr(lse), dt, B, H, Sq, Skv, D, qs.v, ks.v, vs.v, os.v,
                              (float)scale, nullptr, causal, ptr(ws), bytes, stream);
    else
      rc = lib.pa_attn_fwd_narrow(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), (float*)ptr(lse), dt, B, H, Sq, Skv, D, qs.v, ks.v, vs.v, os.v,
                              (float)scale, causal, ptr(ws), bytes, stream);
  }
  if (rc != PA_OK) return PyLong_FromLong(rc);
  return pair(out, lse);
  END_HANDLE_TH_ERRORS
}

bool same_flat(const Tensor& a, const Tensor& b) {
  return plain(b) && b.scalar_type() == a.scalar_type() && b.device() == a.device() && b.sizes() == a.sizes() && b.is_contiguous() &&
         (uintptr_t)b.data_ptr() % 16 == 0;
}
bool flat_operand(const Tensor& a) { return plain(a) && dtype_code(a.scalar_type()) >= 0 && a.numel() > 0 && same_flat(a, a); }

// fbcache_residual(hidden, hidden0, prev or None, step, workspace or None, stream) -> (residual, ratio): against prev, which holds every
// step-th column (the caller has seen to the shapes where step > 1)
PyObject* fbcache_residual(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  const Tensor *h, *h0, *prev, *ws;
  if (nargs != 6 || !optional_tensor(args[0], &h) || !optional_tensor(args[1], &h0) || !optional_tensor(args[2], &prev) || !optional_tensor(args[4], &ws))
    Py_RETURN_NONE;
  const long step = PyLong_AsLong(args[3]);
  void* const stream = PyLong_AsVoidPtr(args[5]);
  if (PyErr_Occurred()) return nullptr;
  if (!h || !h0 || !flat_operand(*h) || !same_flat(*h, *h0)) Py_RETURN_NONE;
  if (prev) {
    if (!ws || !plain(*ws) || !flat_operand(*prev) || prev->scalar_type() != h->scalar_type() || prev->device() != h->device()) Py_RETURN_NONE;
    if (step == 1 ? prev->sizes() != h->sizes() : step < 2 || h->dim() == 0 || prev->numel() * step != h->numel()) Py_RETURN_NONE;
  }
  Tensor resid, ratio;
  int rc;
  {
    pybind11::gil_scoped_release no_gil;
    resid = at::empty(h->sizes(), h->options());
    ratio = at::empty({}, h->options());
    const int dt = dtype_code(h->scalar_type());
    const size_t ws_bytes = prev ? ws->numel() * ws->element_size() : 0;
    if (!prev) rc = lib.pa_fbcache_residual(h->data_ptr(), h0->data_ptr(), resid.data_ptr(), dt, h->numel(), ratio.data_ptr(), stream);
    else if (step == 1)
      rc = lib.pa_fbcache_residual_ratio(h->data_ptr(), h0->data_ptr(), prev->data_ptr(), resid.data_ptr(), dt, h->numel(), ratio.data_ptr(), nullptr,
                                     ws->data_ptr(), ws_bytes, stream);
    else
      rc = lib.pa_fbcache_residual_ratio_strided(h->data_ptr(), h0->data_ptr(), prev->data_ptr(), resid.data_ptr(), dt, h->numel() / h->size(-1), h->size(-1),
                                             (int)step, ratio.data_ptr(), nullptr, ws->data_ptr(), ws_bytes, stream);
  }
  if (rc != PA_OK) return PyLong_FromLong(rc);
  return pair(resid, ratio);
  END_HANDLE_TH_ERRORS
}

// fbcache_apply(residual, hidden, stream) -> residual + hidden
PyObject* fbcache_apply(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  const Tensor *r, *h;
  if (nargs != 3 || !optional_tensor(args[0], &r) || !optional_tensor(args[1], &h) || !r || !h || !flat_operand(*h) || !same_flat(*h, *r)) Py_RETURN_NONE;
  void* const stream = PyLong_AsVoidPtr(args[2]);
  if (PyErr_Occurred()) return nullptr;
  Tensor out;
  int rc;
  {
    pybind11::gil_scoped_release no_gil;
    out = at::empty(h->sizes(), h->options());
    rc = lib.pa_fbcache_apply_residual(r->data_ptr(), h->data_ptr(), out.data_ptr(), dtype_code(h->scalar_type()), h->numel(), stream);
  }
  if (rc != PA_OK) return PyLong_FromLong(rc);
  return THPVariable_Wrap(out);
  END_HANDLE_TH_ERRORS
}

// fbcache_apply_pair(residual, hidden, residual2, hidden2, stream) -> (residual + hidden, residual2 + hidden2)
PyObject* fbcache_apply_pair(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  const Tensor *r, *h, *r2, *h2;
  if (nargs != 5 || !optional_tensor(args[0], &r) || !optional_tensor(args[1], &h) || !optional_tensor(args[2], &r2) || !optional_tensor(args[3], &h2))
    Py_RETURN_NONE;
  if (!r || !h || !r2 || !h2 || !flat_operand(*h) || !flat_operand(*h2) || !same_flat(*h, *r) || !same_flat(*h2, *r2)) Py_RETURN_NONE;
  if (h2->scalar_type() != h->scalar_type() || h2->device() != h->device()) Py_RETURN_NONE;
  void* const stream = PyLong_AsVoidPtr(args[4]);
  if (PyErr_Occurred()) return nullptr;
  Tensor out, out2;
  int rc;
  {
    pybind11::gil_scoped_release no_gil;
    out = at::empty(h->sizes(), h->options());
    out2 = at::empty(h2->sizes(), h2->options());
    rc = lib.pa_fbcache_apply_residual2(r->data_ptr(), h->data_ptr(), out.data_ptr(), h->numel(), r2->data_ptr(), h2->data_ptr(), out2.data_ptr(), h2->numel(),
                                    dtype_code(h->scalar_type()), stream);
  }
  if (rc != PA_OK) return PyLong_FromLong(rc);
  return pair(out, out2);
  END_HANDLE_TH_ERRORS
}

// A sequence of tensors shaped like its first one, which is a flat operand
bool flat_list(PyObject* list, std::vector<const Tensor*>& out) {
  if (!PyList_Check(list) && !PyTuple_Check(list)) return false;
  const Py_ssize_t n = PySequence_Fast_GET_SIZE(list);
  PyObject** items = PySequence_Fast_ITEMS(list);
  for (Py_ssize_t i = 0; i < n; ++i) {
    const Tensor* t;
    if (!optional_tensor(items[i], &t) || !t) return false;
    if (out.empty() ? !flat_operand(*t) : !same_flat(*out[0], *t)) return false;
    out.push_back(t);
  }
  return true;
}

// taylorseer_value(derivs, elapsed, hidden or None, stream) -> value (+ hidden)
PyObject* taylorseer_value(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  std::vector<const Tensor*> d;
  const Tensor* h;
  if (nargs != 4 || !flat_list(args[0], d) || d.empty() || d.size() > 16 || !optional_tensor(args[2], &h) || (h && !same_flat(*d[0], *h))) Py_RETURN_NONE;
  const long elapsed = PyLong_AsLong(args[1]);
  void* const stream = PyLong_AsVoidPtr(args[3]);
  if (PyErr_Occurred()) return nullptr;
  if (elapsed < -65536 || elapsed > 65536) Py_RETURN_NONE;
  const int m = (int)d.size();
  const void* src[16];
  float coef[16], pw[16];
  double factorial = 1, power = 1;  // (exact below 2^53, which is where this path ends)
  for (int i = 0; i < m; ++i) {
    if (i > 0) {
      factorial *= i;
      power *= (double)elapsed;
    }
    if (std::fabs(power) > 9e15) Py_RETURN_NONE;
    src[i] = d[i]->data_ptr();
    coef[i] = (float)(1.0 / factorial);
    pw[i] = (float)power;
  }
  Tensor out;
  int rc;
  {
    pybind11::gil_scoped_release no_gil;
    out = at::empty(d[0]->sizes(), d[0]->options());
    rc = lib.pa_taylorseer_value(src, m, coef, pw, h ? h->data_ptr() : nullptr, out.data_ptr(), dtype_code(out.scalar_type()), out.numel(), stream);
  }
  if (rc != PA_OK) return PyLong_FromLong(rc);
  return THPVariable_Wrap(out);
  END_HANDLE_TH_ERRORS
}

// taylorseer_derivatives(y, prev, window, stream) -> [x1, ..., xn]
PyObject* taylorseer_derivatives(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  std::vector<const Tensor*> d;
  const Tensor* y;
  if (nargs != 4 || !optional_tensor(args[0], &y) || !y || !flat_operand(*y) || !flat_list(args[1], d) || d.empty() || d.size() > 16 || !same_flat(*y, *d[0]))
    Py_RETURN_NONE;
  const double window = PyFloat_AsDouble(args[2]);
  void* const stream = PyLong_AsVoidPtr(args[3]);
  if (PyErr_Occurred()) return nullptr;
  const int n = (int)d.size();
  const void* src[16];
  void* dst[16];
  std::vector<Tensor> cur(n);
  int rc;
  {
    pybind11::gil_scoped_release no_gil;
    for (int i = 0; i < n; ++i) {
      cur[i] = at::empty(y->sizes(), y->options());
      src[i] = d[i]->data_ptr();
      dst[i] = cur[i].data_ptr();
    }
    rc = lib.pa_taylorseer_update(y->data_ptr(), src, dst, n, dtype_code(y->scalar_type()), y->numel(), (float)window, stream);
  }
  if (rc != PA_OK) return PyLong_FromLong(rc);
  PyObject* list = PyList_New(n);
  if (!list) return nullptr;
  for (int i = 0; i < n; ++i) PyList_SET_ITEM(list, i, THPVariable_Wrap(cur[i]));
  return list;
  END_HANDLE_TH_ERRORS
}

// block_sparse(query, key, value, block_mask, scale or None, stream) -> (out, lse): the mask covers all rows and keys
PyObject* block_sparse(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  const Tensor *pq, *pk, *pv, *m;
  if (nargs != 6 || !optional_tensor(args[0], &pq) || !optional_tensor(args[1], &pk) || !optional_tensor(args[2], &pv) || !optional_tensor(args[3], &m))
    Py_RETURN_NONE;
  if (!pq || !pk || !pv || !m || !attention_operands(*pq, *pk, *pv)) Py_RETURN_NONE;
  const Tensor &q = *pq, &k = *pk, &v = *pv;
  const int64_t B = q.size(0), H = q.size(1), Sq = q.size(2), D = q.size(3), Skv = k.size(2);
  if (B > INT32_MAX || H > INT32_MAX || Sq > INT32_MAX || Skv > INT32_MAX || (D != 64 && D != 128)) Py_RETURN_NONE;
  if (!plain(*m) || m->device() != q.device() || m->scalar_type() != at::kBool || m->dim() < 2 || m->dim() > 3 || !m->is_contiguous()) Py_RETURN_NONE;
  const int64_t Hm = m->dim() == 3 ? m->size(0) : 1, nQ = m->size(-2), nK = m->size(-1);
  if ((Hm != 1 && Hm != H) || nQ <= 0 || nK <= 0 || nQ > Sq || nK > Skv || Sq % nQ != 0 || Skv % nK != 0) Py_RETURN_NONE;
  double scale = 1.0 / std::sqrt((double)D);
  if (args[4] != Py_None) scale = PyFloat_AsDouble(args[4]);
  void* const stream = PyLong_AsVoidPtr(args[5]);
  if (PyErr_Occurred()) return nullptr;
  const Strides3 qs(q), ks(k), vs(v);
  Tensor out, lse;
  int rc;
  {
    pybind11::gil_scoped_release no_gil;
    const size_t bytes = lib.pa_blocksparse_workspace_bytes((int)Hm, (int)nQ, (int)nK);
    out = out_like(q);
    lse = at::empty({B, H, Sq}, q.options().dtype(at::kFloat));
    const Tensor ws = scratch((bytes + 3) / 4 * 4, q);
    const Strides3 os(out);
    rc = lib.pa_attn_fwd_blocksparse(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), (float*)lse.data_ptr(), dtype_code(q.scalar_type()), B, H, Sq, Skv,
                                 D, qs.v, ks.v, vs.v, os.v, (float)scale, (const uint8_t*)m->data_ptr(), (int)Hm, (int)nQ, (int)nK, 0, (int)(Sq / nQ), 0,
                                 (int)(Skv / nK), (int32_t*)ptr(ws), bytes, stream);
  }
  if (rc != PA_OK) return PyLong_FromLong(rc);
  return pair(out, lse);
  END_HANDLE_TH_ERRORS
}

#define METHOD(name) {#name, (PyCFunction)(void (*)(void))name, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {{"bind", bind, METH_O, nullptr},
                         METHOD(attention),        METHOD(block_sparse),     METHOD(fbcache_residual),       METHOD(fbcache_apply),
                         METHOD(fbcache_apply_pair), METHOD(taylorseer_value), METHOD(taylorseer_derivatives), {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host_calls", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host_calls(void) {
  PyObject* const m = PyModule_Create(&module);
  if (m && PyModule_AddStringConstant(m, "torch_version", BUILT_WITH_TORCH) < 0) {  // whose C++ interface this is
    Py_DECREF(m);
    return nullptr;
  }
  return m;
}
