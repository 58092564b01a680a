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
#include <torch/version.h>

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

// A torch C++ exception before the launch (an allocation that fails, a tensor
// without storage): the Python path takes the call and raises its own error
// (torch.OutOfMemoryError, not a plain RuntimeError).
PyObject* declined() {
  PyErr_Clear();
  Py_RETURN_NONE;
}

// Every torch call that can throw (data_ptr() of a tensor without storage
// among them) comes before a launch, with the interpreter lock held; Unlocked
// covers the library call alone.
struct Unlocked {
  PyThreadState* state = PyEval_SaveThread();
  Unlocked() = default;
  Unlocked(const Unlocked&) = delete;
  ~Unlocked() { PyEval_RestoreThread(state); }
};

// A tensor of a call as the library takes it.
struct Rows {
  void* p = nullptr;
  int64_t s0 = 0, s1 = 0;
};
Rows rows(const at::Tensor* t) {
  return t != nullptr && t->defined() ? Rows{t->data_ptr(), t->stride(0), t->stride(1)} : Rows{};
}
void* address(const at::Tensor* t) { return t != nullptr ? t->data_ptr() : nullptr; }

// A new reference to `t` after a launch: an error here is raised, the call is
// not made again.
PyObject* wrap(at::Tensor&& t) {
  try {
    return THPVariable_Wrap(std::move(t));
  } catch (const std::exception& e) {
    if (!PyErr_Occurred()) PyErr_SetString(PyExc_RuntimeError, e.what());
    return nullptr;
  }
}

// decode(out or None, q, k_cache, v_cache, block_tables, context_lens, scale,
//        stream, key or None, value, slot_mapping)
PyObject* decode(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 11) {
    PyErr_SetString(PyExc_TypeError, "decode takes 11 arguments");
    return nullptr;
  }
  at::Tensor out, ws;
  Rows q_r, k_r, v_r, out_r;
  void *slots_p, *kc_p, *vc_p, *bt_p, *lens_p, *ws_p, *stream;
  int64_t batch, heads, kvh, pages, page, bt_stride, blocks;
  size_t bytes;
  float scale;
  int sb = 4;
  const bool append = a[8] != Py_None;
  try {
    const at::Tensor* q = tensor(a[1]);
    if (q == nullptr || !q->defined() || !plain(q, at::kBFloat16, 3, *q)) Py_RETURN_NONE;
    const at::Tensor *kc = tensor(a[2]), *vc = tensor(a[3]), *bt = tensor(a[4]),
                     *lens = tensor(a[5]);
    if (!decode_shapes(*q, kc, vc, bt, lens) || !PyFloat_CheckExact(a[6])) Py_RETURN_NONE;
    batch = q->size(0), heads = q->size(1), kvh = kc->size(2);
    pages = kc->size(0), page = kc->size(1), bt_stride = bt->stride(0), blocks = bt->size(1);
    const at::Tensor *key = nullptr, *value = nullptr, *slots = nullptr;
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
    if (a[0] != Py_None) {
      const at::Tensor* given = tensor(a[0]);
      if (!plain(given, at::kBFloat16, 3, *q) || given->sizes() != q->sizes() ||
          given->stride(2) != 1)
        Py_RETURN_NONE;
      out = *given;
    } else {
      out = output_like(*q);
    }
    stream = PyLong_AsVoidPtr(a[7]);
    if (PyErr_Occurred()) return nullptr;
    scale = float(PyFloat_AS_DOUBLE(a[6]));
    bytes = p_workspace(batch, heads, kvh, 128, page, blocks);
    if (bytes > 0) ws = at::empty({int64_t(bytes)}, q->options().dtype(at::kByte));
    ws_p = bytes > 0 ? ws.data_ptr() : nullptr;
    q_r = rows(q), k_r = rows(key), v_r = rows(value), out_r = rows(&out);
    slots_p = address(slots);
    kc_p = address(kc), vc_p = address(vc), bt_p = address(bt), lens_p = address(lens);
  } catch (const std::exception&) {
    return declined();
  }
  int rc;
  if (append) {
    Unlocked unlocked;
    rc = p_decode_append(q_r.p, q_r.s0, q_r.s1, k_r.p, k_r.s0, k_r.s1, v_r.p, v_r.s0, v_r.s1,
                         slots_p, sb, kc_p, vc_p, pages, page, kvh, 128,
                         static_cast<const int32_t*>(bt_p), bt_stride, blocks,
                         static_cast<const int32_t*>(lens_p), batch, heads, scale, out_r.p,
                         out_r.s0, out_r.s1, ws_p, bytes, stream);
  } else {
    Unlocked unlocked;
    rc = p_decode(q_r.p, q_r.s0, q_r.s1, kc_p, vc_p, pages, page, kvh, 128, KVC_KV_BF16, nullptr,
                  nullptr, nullptr, nullptr, nullptr, nullptr, 0,
                  static_cast<const int32_t*>(bt_p), bt_stride, blocks,
                  static_cast<const int32_t*>(lens_p), batch, heads, scale, out_r.p, out_r.s0,
                  out_r.s1, ws_p, bytes, stream);
  }
  if (rc != KVC_OK) return fail(rc, "paged_decode");
  if (a[0] != Py_None) {
    Py_INCREF(a[0]);
    return a[0];
  }
  return wrap(std::move(out));
}

// rope(q, k, v or None, positions, cos_sin, q_weight or None, k_weight or
//      None, eps, k_cache or None, v_cache, slot_mapping, return_k, stream)
PyObject* rope(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 13) {
    PyErr_SetString(PyExc_TypeError, "rope takes 13 arguments");
    return nullptr;
  }
  at::Tensor q_out, k_out;
  Rows q_r, k_r, v_r, qo_r, ko_r;
  void *pos_p, *cs_p, *qw_p, *kw_p, *kc_p, *vc_p, *slots_p, *stream;
  int64_t tokens, heads, kvh, max_position, num_slots = 0;
  int pb = 4, sb = 4;
  float eps;
  try {
    const at::Tensor *q = tensor(a[0]), *k = tensor(a[1]), *pos = tensor(a[3]),
                     *cs = tensor(a[4]);
    if (q == nullptr || !q->defined() || !plain(q, at::kBFloat16, 3, *q) ||
        !plain(k, at::kBFloat16, 3, *q) || !plain(cs, at::kFloat, 2, *q))
      Py_RETURN_NONE;
    tokens = q->size(0), heads = q->size(1), kvh = k->size(1);
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
    const at::Tensor *kc = nullptr, *vc = nullptr, *slots = nullptr;
    if (a[8] != Py_None) {
      kc = tensor(a[8]);
      vc = tensor(a[9]);
      slots = tensor(a[10]);
      if (v == nullptr || !plain(kc, at::kBFloat16, 4, *q) || !plain(vc, at::kBFloat16, 4, *q) ||
          kc->sizes() != vc->sizes() || !kc->is_contiguous() || !vc->is_contiguous() ||
          !is_index(slots, tokens, *q, &sb))
        Py_RETURN_NONE;
      num_slots = kc->numel() / (kvh * 128);
    } else if (a[9] != Py_None) {
      Py_RETURN_NONE;  // a v pool alone is refused
    }
    stream = PyLong_AsVoidPtr(a[12]);
    if (PyErr_Occurred()) return nullptr;
    eps = float(PyFloat_AS_DOUBLE(a[7]));
    max_position = cs->size(0);
    q_out = at::empty({tokens, heads, 128}, q->options());
    if (a[11] == Py_True) k_out = at::empty({tokens, kvh, 128}, k->options());
    q_r = rows(q), k_r = rows(k), v_r = rows(v), qo_r = rows(&q_out), ko_r = rows(&k_out);
    pos_p = address(pos), cs_p = address(cs), qw_p = address(w[0]), kw_p = address(w[1]);
    kc_p = address(kc), vc_p = address(vc), slots_p = address(slots);
  } catch (const std::exception&) {
    return declined();
  }
  int rc;
  {
    Unlocked unlocked;
    rc = p_rope(q_r.p, q_r.s0, q_r.s1, k_r.p, k_r.s0, k_r.s1, v_r.p, v_r.s0, v_r.s1, tokens,
                heads, kvh, 128, pos_p, pb, qw_p, kw_p, eps, static_cast<const float*>(cs_p),
                max_position, qo_r.p, qo_r.s0, qo_r.s1, ko_r.p, ko_r.s0, ko_r.s1, kc_p, vc_p,
                num_slots, slots_p, sb, stream);
  }
  if (rc != KVC_OK) return fail(rc, "kvc_qk_norm_rope_store");
  PyObject* r = PyTuple_New(2);
  if (r == nullptr) return nullptr;
  PyObject* q_py = wrap(std::move(q_out));
  PyObject* k_py = nullptr;
  if (ko_r.p != nullptr) {
    k_py = wrap(std::move(k_out));
  } else {
    Py_INCREF(Py_None);
    k_py = Py_None;
  }
  PyTuple_SET_ITEM(r, 0, q_py);
  PyTuple_SET_ITEM(r, 1, k_py);
  if (q_py != nullptr && k_py != nullptr) return r;
  Py_DECREF(r);
  return nullptr;
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

PyMODINIT_FUNC PyInit__kvc_host() {
  PyObject* m = PyModule_Create(&module);
  if (m != nullptr && PyModule_AddStringConstant(m, "torch_version", TORCH_VERSION) < 0) {
    Py_DECREF(m);
    return nullptr;
  }
  return m;
}
