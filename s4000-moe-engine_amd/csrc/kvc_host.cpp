// Native host path of the decode step's calls.
//
// A decode step at a small batch is shorter on the GPU (14-20 us) than its
// Python call was on the host (20-31 us): the argument checks, the output and
// workspace allocations and a 34-argument ctypes call.  This extension does
// the same work for the form such a step has (exact torch.Tensor arguments on
// one GPU, bf16, the strides and index types the launch reads as they are)
// and returns None, having done nothing, for anything else: the Python
// function then checks, converts or raises as it always did.  Nothing is
// kept between calls.  Measured: one row of 333 tokens through norm, rotary,
// append and attention (16 q / 8 kv heads) 30 -> 16-18 us a pass, a decode
// step of 11 rows of 97-1501 tokens 20.0 -> 14.7 us (both now GPU-bound).
#include <Python.h>

#include <ATen/ATen.h>
#include <dlfcn.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstdlib>
#include <cstring>

#include "kvc.h"

namespace {

decltype(&kvc_last_error) p_last_error;
decltype(&kvc_paged_decode_workspace_bytes) p_workspace;
decltype(&kvc_paged_decode) p_decode;
decltype(&kvc_paged_decode_append) p_decode_append;
decltype(&kvc_qk_norm_rope_store) p_rope;

// The tensor behind an exact torch.Tensor / Parameter, else null.
const at::Tensor* tensor(PyObject* o) {
  return THPVariable_CheckExact(o) ? &THPVariable_Unpack(o) : nullptr;
}

// A plain dense-storage tensor of `type` on `like`'s GPU with `dim` dims.
bool plain(const at::Tensor* t, at::ScalarType type, int64_t dim, const at::Tensor& like) {
  return t != nullptr && t->defined() && t->is_cuda() && t->layout() == at::kStrided &&
         t->scalar_type() == type && t->dim() == dim && t->device() == like.device();
}

bool is_index(const at::Tensor* t, int64_t n, const at::Tensor& like, int* bytes) {
  if (t == nullptr || !t->defined() || t->dim() != 1 || t->numel() != n || !t->is_contiguous())
    return false;
  *bytes = t->scalar_type() == at::kLong ? 8 : 4;
  return plain(t, *bytes == 8 ? at::kLong : at::kInt, 1, like);
}

// [pages, page, kv heads, 128] pools of a decode over q [batch, heads, 128].
bool decode_shapes(const at::Tensor& q, const at::Tensor* kc, const at::Tensor* vc,
                   const at::Tensor* bt, const at::Tensor* lens) {
  if (!plain(kc, at::kBFloat16, 4, q) || !plain(vc, at::kBFloat16, 4, q) ||
      !plain(bt, at::kInt, 2, q) || !plain(lens, at::kInt, 1, q))
    return false;
  const int64_t page = kc->size(1), kvh = kc->size(2);
  return q.size(0) > 0 && q.size(2) == 128 && q.stride(2) == 1 && kc->sizes() == vc->sizes() &&
         kc->size(3) == 128 && kvh > 0 && q.size(1) > 0 && q.size(1) % kvh == 0 && page > 0 &&
         page % 32 == 0 && kc->is_contiguous() && vc->is_contiguous() && bt->stride(1) == 1 &&
         bt->size(0) >= q.size(0) && bt->size(1) > 0 && lens->is_contiguous() &&
         lens->numel() >= q.size(0);
}

at::Tensor output_like(const at::Tensor& q) {
  at::Tensor out = at::empty_like(q);
  return out.stride(2) == 1 ? out : at::empty(q.sizes(), q.options());
}

// nullptr with the exception _native.call raises for the status.
PyObject* fail(int rc, const char* what) {
  const char* msg = p_last_error();
  PyObject* type = rc == KVC_ERR_ASSERT ? PyExc_AssertionError
                   : rc == KVC_ERR_RUNTIME || (rc != KVC_ERR_VALUE && rc != KVC_ERR_WORKSPACE)
                       ? PyExc_RuntimeError
                       : PyExc_ValueError;
  if (msg != nullptr && *msg != '\0') {
    PyErr_SetString(type, msg);
  } else {
    PyErr_Format(type, "%s failed with status %d", what, rc);
  }
  return nullptr;
}

// A torch C++ exception (an allocation that fails, a tensor without storage):
// nothing has been launched, so the Python path takes the call and raises its
// own error (torch.OutOfMemoryError, not a plain RuntimeError).
PyObject* declined() {
  PyErr_Clear();
  Py_RETURN_NONE;
}

// decode(out or None, q, k_cache, v_cache, block_tables, context_lens, scale,
//        stream, key or None, value, slot_mapping)
PyObject* decode(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 11) {
    PyErr_SetString(PyExc_TypeError, "decode takes 11 arguments");
    return nullptr;
  }
  try {
    const at::Tensor* q = tensor(a[1]);
    if (q == nullptr || !q->defined() || !plain(q, at::kBFloat16, 3, *q)) Py_RETURN_NONE;
    const at::Tensor *kc = tensor(a[2]), *vc = tensor(a[3]), *bt = tensor(a[4]),
                     *lens = tensor(a[5]);
    if (!decode_shapes(*q, kc, vc, bt, lens) || !PyFloat_CheckExact(a[6])) Py_RETURN_NONE;
    const int64_t batch = q->size(0), heads = q->size(1), kvh = kc->size(2);
    const bool append = a[8] != Py_None;
    const at::Tensor *key = nullptr, *value = nullptr, *slots = nullptr;
    int sb = 4;
    if (append) {
      key = tensor(a[8]);
      value = tensor(a[9]);
      slots = tensor(a[10]);
      const char* check = std::getenv("KVC_CHECK_APPEND");
      if (!plain(key, at::kBFloat16, 3, *q) || !plain(value, at::kBFloat16, 3, *q) ||
          key->sizes() != value->sizes() || key->size(0) != batch || key->size(1) != kvh ||
          key->size(2) != 128 || key->stride(2) != 1 || value->stride(2) != 1 ||
          !is_index(slots, batch, *q, &sb) || (check != nullptr && std::strcmp(check, "1") == 0))
        Py_RETURN_NONE;
    }
    at::Tensor out;
    if (a[0] != Py_None) {
      const at::Tensor* given = tensor(a[0]);
      if (!plain(given, at::kBFloat16, 3, *q) || given->sizes() != q->sizes() ||
          given->stride(2) != 1)
        Py_RETURN_NONE;
      out = *given;
    } else {
      out = output_like(*q);
    }
    void* stream = PyLong_AsVoidPtr(a[7]);
    if (PyErr_Occurred()) return nullptr;
    const float scale = float(PyFloat_AS_DOUBLE(a[6]));
    const size_t bytes = p_workspace(batch, heads, kvh, 128, kc->size(1), bt->size(1));
    at::Tensor ws;
    if (bytes > 0) ws = at::empty({int64_t(bytes)}, q->options().dtype(at::kByte));
    void* wp = bytes > 0 ? ws.data_ptr() : nullptr;
    int rc;
    Py_BEGIN_ALLOW_THREADS;
    if (append) {
      rc = p_decode_append(q->data_ptr(), q->stride(0), q->stride(1), key->data_ptr(),
                           key->stride(0), key->stride(1), value->data_ptr(), value->stride(0),
                           value->stride(1), slots->data_ptr(), sb, kc->data_ptr(),
                           vc->data_ptr(), kc->size(0), kc->size(1), kvh, 128,
                           static_cast<const int32_t*>(bt->data_ptr()), bt->stride(0),
                           bt->size(1), static_cast<const int32_t*>(lens->data_ptr()), batch,
                           heads, scale, out.data_ptr(), out.stride(0), out.stride(1), wp, bytes,
                           stream);
    } else {
      rc = p_decode(q->data_ptr(), q->stride(0), q->stride(1), kc->data_ptr(), vc->data_ptr(),
                    kc->size(0), kc->size(1), kvh, 128, KVC_KV_BF16, nullptr, nullptr, nullptr,
                    nullptr, nullptr, nullptr, 0, static_cast<const int32_t*>(bt->data_ptr()),
                    bt->stride(0), bt->size(1), static_cast<const int32_t*>(lens->data_ptr()),
                    batch, heads, scale, out.data_ptr(), out.stride(0), out.stride(1), wp, bytes,
                    stream);
    }
    Py_END_ALLOW_THREADS;
    if (rc != KVC_OK) return fail(rc, "paged_decode");
    if (a[0] != Py_None) {
      Py_INCREF(a[0]);
      return a[0];
    }
    return THPVariable_Wrap(std::move(out));
  } catch (const std::exception&) {
    return declined();
  }
}

// rope(q, k, v or None, positions, cos_sin, q_weight or None, k_weight or
//      None, eps, k_cache or None, v_cache, slot_mapping, return_k, stream)
PyObject* rope(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 13) {
    PyErr_SetString(PyExc_TypeError, "rope takes 13 arguments");
    return nullptr;
  }
  try {
    const at::Tensor *q = tensor(a[0]), *k = tensor(a[1]), *pos = tensor(a[3]),
                     *cs = tensor(a[4]);
    if (q == nullptr || !q->defined() || !plain(q, at::kBFloat16, 3, *q) ||
        !plain(k, at::kBFloat16, 3, *q) || !plain(cs, at::kFloat, 2, *q))
      Py_RETURN_NONE;
    const int64_t tokens = q->size(0), heads = q->size(1), kvh = k->size(1);
    int pb = 4, sb = 4;
    if (tokens == 0 || q->size(2) != 128 || k->size(0) != tokens || k->size(2) != 128 ||
        kvh == 0 || heads == 0 || q->stride(2) != 1 || k->stride(2) != 1 || cs->size(1) != 128 ||
        !cs->is_contiguous() || !is_index(pos, tokens, *q, &pb) || !PyFloat_CheckExact(a[7]) ||
        (a[11] != Py_True && a[11] != Py_False))
      Py_RETURN_NONE;
    const at::Tensor* w[2] = {nullptr, nullptr};
    for (int i = 0; i < 2; ++i) {
      if (a[5 + i] == Py_None) continue;
      w[i] = tensor(a[5 + i]);
      if (!plain(w[i], at::kBFloat16, 1, *q) || w[i]->size(0) != 128 || !w[i]->is_contiguous())
        Py_RETURN_NONE;
    }
    const at::Tensor* v = nullptr;
    if (a[2] != Py_None) {
      v = tensor(a[2]);
      if (!plain(v, at::kBFloat16, 3, *q) || v->sizes() != k->sizes() || v->stride(2) != 1)
        Py_RETURN_NONE;
    }
    const bool cache = a[8] != Py_None;
    const at::Tensor *kc = nullptr, *vc = nullptr, *slots = nullptr;
    if (cache) {
      kc = tensor(a[8]);
      vc = tensor(a[9]);
      slots = tensor(a[10]);
      if (v == nullptr || !plain(kc, at::kBFloat16, 4, *q) || !plain(vc, at::kBFloat16, 4, *q) ||
          kc->sizes() != vc->sizes() || !kc->is_contiguous() || !vc->is_contiguous() ||
          !is_index(slots, tokens, *q, &sb))
        Py_RETURN_NONE;
    }
    void* stream = PyLong_AsVoidPtr(a[12]);
    if (PyErr_Occurred()) return nullptr;
    const float eps = float(PyFloat_AS_DOUBLE(a[7]));
    at::Tensor q_out = at::empty({tokens, heads, 128}, q->options());
    at::Tensor k_out;
    if (a[11] == Py_True) k_out = at::empty({tokens, kvh, 128}, k->options());
    const bool ko = k_out.defined();
    int rc;
    Py_BEGIN_ALLOW_THREADS;
    rc = p_rope(q->data_ptr(), q->stride(0), q->stride(1), k->data_ptr(), k->stride(0),
                k->stride(1), v != nullptr ? v->data_ptr() : nullptr,
                v != nullptr ? v->stride(0) : 0, v != nullptr ? v->stride(1) : 0, tokens, heads,
                kvh, 128, pos->data_ptr(), pb, w[0] != nullptr ? w[0]->data_ptr() : nullptr,
                w[1] != nullptr ? w[1]->data_ptr() : nullptr, eps,
                static_cast<const float*>(cs->data_ptr()), cs->size(0), q_out.data_ptr(),
                q_out.stride(0), q_out.stride(1), ko ? k_out.data_ptr() : nullptr,
                ko ? k_out.stride(0) : 0, ko ? k_out.stride(1) : 0,
                cache ? kc->data_ptr() : nullptr, cache ? vc->data_ptr() : nullptr,
                cache ? kc->numel() / (kvh * 128) : 0, cache ? slots->data_ptr() : nullptr, sb,
                stream);
    Py_END_ALLOW_THREADS;
    if (rc != KVC_OK) return fail(rc, "kvc_qk_norm_rope_store");
    PyObject* r = PyTuple_New(2);
    if (r == nullptr) return nullptr;
    PyTuple_SET_ITEM(r, 0, THPVariable_Wrap(std::move(q_out)));
    if (ko) {
      PyTuple_SET_ITEM(r, 1, THPVariable_Wrap(std::move(k_out)));
    } else {
      Py_INCREF(Py_None);
      PyTuple_SET_ITEM(r, 1, Py_None);
    }
    return r;
  } catch (const std::exception&) {
    return declined();
  }
}

template <typename F>
bool resolve(void* lib, const char* name, F& fn) {
  fn = reinterpret_cast<F>(dlsym(lib, name));
  if (fn == nullptr) PyErr_Format(PyExc_RuntimeError, "%s is not in the kvc library", name);
  return fn != nullptr;
}

// bind(path): the library at `path` (already loaded by _native).
PyObject* bind(PyObject*, PyObject* path) {
  const char* p = PyUnicode_AsUTF8(path);
  if (p == nullptr) return nullptr;
  void* lib = dlopen(p, RTLD_NOW);
  if (lib == nullptr) {
    PyErr_Format(PyExc_RuntimeError, "cannot open %s: %s", p, dlerror());
    return nullptr;
  }
  if (!resolve(lib, "kvc_last_error", p_last_error) ||
      !resolve(lib, "kvc_paged_decode_workspace_bytes", p_workspace) ||
      !resolve(lib, "kvc_paged_decode", p_decode) ||
      !resolve(lib, "kvc_paged_decode_append", p_decode_append) ||
      !resolve(lib, "kvc_qk_norm_rope_store", p_rope))
    return nullptr;
  Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"bind", bind, METH_O, "bind(path): resolve the kvc entry points"},
    {"decode", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(decode)), METH_FASTCALL,
     "one paged decode (with the step's append when a key is given), or None"},
    {"rope", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(rope)), METH_FASTCALL,
     "the fused norm, rotary and append, or None"},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_kvc_host", nullptr, -1, methods,
                      nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__kvc_host() { return PyModule_Create(&module); }
