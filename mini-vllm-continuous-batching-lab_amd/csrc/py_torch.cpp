// _mvtorch: the per-layer launches of an eager step from the step's packed
// words and the layer's tensors, with the wrappers' per-call checks, in native
// code (host C++ on torch's tensor API, no HIP).
//
// A small layer's call is bound by its launch: in Python the checks, the
// pointers and strides, the output's allocation and the step's cache lookups
// take 8-15 us of host time around a launch of 3 us, where the kernels of a
// short decode or prompt take 4-10. Every function here checks what the Python
// wrapper checks and returns None where anything differs from the plain case
// (other shapes, types, devices, strides or alignments, subclassed tensors): the
// wrapper then runs its own path, which makes the copies or raises. Otherwise
// it launches and returns the outputs, or the entry point's status code where
// that is not 0. Nothing is kept between calls.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <ATen/ATen.h>

#include <cstdint>
#include <cstring>

#include "mvattn.h"

namespace {

decltype(&mv_paged_decode_write) g_decode_write;
decltype(&mv_paged_decode) g_decode;
decltype(&mv_kv_cache_write) g_cache_write;
decltype(&mv_rope_kv_cache_write) g_rope_write;
decltype(&mv_paged_prefill_blocks) g_prefill;

int dtype_code(at::ScalarType t) {
  switch (t) {
    case at::kFloat: return MV_DTYPE_F32;
    case at::kHalf: return MV_DTYPE_F16;
    case at::kBFloat16: return MV_DTYPE_BF16;
    default: return -1;
  }
}

const at::Tensor* plain(PyObject* o) {  // a torch.Tensor, no subclass
  return THPVariable_CheckExact(o) ? &THPVariable_Unpack(o) : nullptr;
}

bool sized(const at::Tensor& t, std::initializer_list<int64_t> s) {
  return t.sizes() == at::IntArrayRef(s.begin(), s.size());
}

// [T, H, D] rows as the kernels read them: D contiguous, 16-byte aligned.
struct Rows {
  void* p;
  int64_t st, sh;
};
bool aligned_rows(const at::Tensor& t, Rows& r) {
  const int64_t eb = t.element_size();
  r = {t.data_ptr(), t.stride(0), t.stride(1)};
  return t.stride(2) == 1 && r.st * eb % 16 == 0 && r.sh * eb % 16 == 0 &&
         reinterpret_cast<uintptr_t>(r.p) % 16 == 0;
}

// The two caches of one layer: the pool layout, contiguous, of `like`'s type and device.
bool caches_ok(const at::Tensor& kc, const at::Tensor& vc, const at::Tensor& like) {
  return kc.dim() == 4 && kc.sizes() == vc.sizes() && kc.scalar_type() == like.scalar_type() &&
         vc.scalar_type() == like.scalar_type() && kc.device() == like.device() &&
         vc.device() == like.device() && kc.is_contiguous() && vc.is_contiguous();
}

PyObject* none() { Py_RETURN_NONE; }
PyObject* status(int rc) { return PyLong_FromLong(rc); }
void* address(PyObject* o) { return o == Py_None ? nullptr : PyLong_AsVoidPtr(o); }

// A step's packed words (the layouts are _hip.py's): little-endian 64-bit
// integers, a double where noted.
struct Words {
  const char* p = nullptr;
  Words(PyObject* o, Py_ssize_t count) {
    char* b;
    Py_ssize_t n;
    if (PyBytes_AsStringAndSize(o, &b, &n) == 0 && n == 8 * count) p = b;
    PyErr_Clear();
  }
  int64_t i(int k) const {
    int64_t v;
    std::memcpy(&v, p + 8 * k, 8);
    return v;
  }
  double f(int k) const {
    double v;
    std::memcpy(&v, p + 8 * k, 8);
    return v;
  }
  template <class T>
  T* ptr(int k) const { return reinterpret_cast<T*>(i(k)); }
};

// seen(refs, versions, tensor, ...): the tensors are the live objects of the
// weak references, at these in-place versions.
PyObject* seen(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n < 2 || !PyTuple_Check(a[0]) || !PyTuple_Check(a[1]) || PyTuple_GET_SIZE(a[0]) != n - 2 ||
      PyTuple_GET_SIZE(a[1]) != n - 2)
    Py_RETURN_FALSE;
  for (Py_ssize_t k = 0; k < n - 2; ++k) {
    PyObject* t = a[k + 2];
    if (!THPVariable_Check(t) || PyWeakref_GetObject(PyTuple_GET_ITEM(a[0], k)) != t) Py_RETURN_FALSE;
    const at::Tensor& x = THPVariable_Unpack(t);
    if (x.is_inference()) Py_RETURN_FALSE;  // (no version: the Python comparison decides)
    if (static_cast<int64_t>(x._version()) != PyLong_AsLongLong(PyTuple_GET_ITEM(a[1], k))) Py_RETURN_FALSE;
  }
  Py_RETURN_TRUE;
  END_HANDLE_TH_ERRORS
}

// decode_write(step words, query, key_cache, value_cache, block_table, kv_len,
// block_size, new_key, new_value, positions or None, device index, stream)
PyObject* decode_write(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 12) return PyErr_Format(PyExc_TypeError, "_mvtorch.decode_write takes 12 arguments");
  const Words w(a[0], 20);
  const at::Tensor *q = plain(a[1]), *kc = plain(a[2]), *vc = plain(a[3]), *bt = plain(a[4]), *kv = plain(a[5]),
                   *nk = plain(a[7]), *nv = plain(a[8]);
  const at::Tensor* pos = a[9] == Py_None ? nullptr : plain(a[9]);
  if (!w.p || !q || !kc || !vc || !bt || !kv || !nk || !nv || (a[9] != Py_None && !pos)) return none();
  const int64_t b = w.i(11), hq = w.i(12), hkv = w.i(13), d = w.i(14), bs = w.i(15), nb = w.i(16);
  const int64_t block_size = PyLong_AsLongLong(a[6]), device = PyLong_AsLongLong(a[10]);
  if (PyErr_Occurred()) return nullptr;
  Rows rq, rk, rv;
  if (block_size != bs || !q->is_cuda() || q->device().index() != device || dtype_code(q->scalar_type()) != w.i(17) ||
      !sized(*q, {b, hq, d}) || !sized(*nk, {b, hkv, d}) || !sized(*nv, {b, hkv, d}) ||
      nk->scalar_type() != q->scalar_type() || nv->scalar_type() != q->scalar_type() || nk->device() != q->device() ||
      nv->device() != q->device() || !caches_ok(*kc, *vc, *q) || !sized(*kc, {nb, hkv, bs, d}) || bt->dim() < 1 ||
      bt->size(0) != b || !sized(*kv, {b}) || (pos && !sized(*pos, {b})) || b == 0 || !aligned_rows(*q, rq) ||
      !aligned_rows(*nk, rk) || !aligned_rows(*nv, rv))
    return none();
  at::Tensor out = at::empty({b, hq, d}, q->options());
  const int rc = g_decode_write(
      rq.p, rq.st, rq.sh, rk.p, rk.st, rk.sh, rv.p, rv.st, rv.sh, w.ptr<const int64_t>(0), w.ptr<const void>(1),
      w.ptr<const void>(2), kc->data_ptr(), vc->data_ptr(), w.ptr<const int32_t>(3), w.ptr<const int32_t>(4), w.i(5),
      static_cast<int32_t>(w.i(6)), static_cast<int32_t>(w.i(7)), static_cast<int32_t>(w.i(8)), w.ptr<int32_t>(9),
      out.data_ptr(), hq * d, d, static_cast<float>(w.f(10)), static_cast<int32_t>(b), static_cast<int32_t>(hq),
      static_cast<int32_t>(hkv), static_cast<int32_t>(d), static_cast<int32_t>(bs), nb, static_cast<int32_t>(w.i(17)),
      w.ptr<void>(18), static_cast<size_t>(w.i(19)), address(a[11]));
  return rc ? status(rc) : THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// decode(plan words, query, key_cache, value_cache, block_table, kv_len,
// block_size, device index, stream)
PyObject* decode(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 9) return PyErr_Format(PyExc_TypeError, "_mvtorch.decode takes 9 arguments");
  const Words w(a[0], 17);
  const at::Tensor *q = plain(a[1]), *kc = plain(a[2]), *vc = plain(a[3]), *bt = plain(a[4]), *kv = plain(a[5]);
  if (!w.p || !q || !kc || !vc || !bt || !kv) return none();
  const int64_t b = w.i(8), hq = w.i(9), hkv = w.i(10), d = w.i(11), bs = w.i(12), nb = w.i(13);
  const int64_t block_size = PyLong_AsLongLong(a[6]), device = PyLong_AsLongLong(a[7]);
  if (PyErr_Occurred()) return nullptr;
  Rows rq;
  if (block_size != bs || !q->is_cuda() || q->device().index() != device || dtype_code(q->scalar_type()) != w.i(14) ||
      !sized(*q, {b, hq, d}) || !caches_ok(*kc, *vc, *q) || !sized(*kc, {nb, hkv, bs, d}) || bt->dim() < 1 ||
      bt->size(0) != b || !sized(*kv, {b}) || b == 0 || !aligned_rows(*q, rq))
    return none();
  at::Tensor out = at::empty({b, hq, d}, q->options());
  const int rc = g_decode(rq.p, rq.st, rq.sh, kc->data_ptr(), vc->data_ptr(), w.ptr<const int32_t>(0),
                          w.ptr<const int32_t>(1), w.i(2), static_cast<int32_t>(w.i(3)), static_cast<int32_t>(w.i(4)),
                          static_cast<int32_t>(w.i(5)), w.ptr<int32_t>(6), out.data_ptr(), hq * d, d,
                          static_cast<float>(w.f(7)), static_cast<int32_t>(b), static_cast<int32_t>(hq),
                          static_cast<int32_t>(hkv), static_cast<int32_t>(d), static_cast<int32_t>(bs), nb,
                          static_cast<int32_t>(w.i(14)), w.ptr<void>(15), static_cast<size_t>(w.i(16)), address(a[8]));
  return rc ? status(rc) : THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// cache_write(checked slots, total slots they were checked for, key, value,
// key_cache, value_cache, slot_mapping as given, block_size, stream):
// True when launched
PyObject* cache_write(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 9) return PyErr_Format(PyExc_TypeError, "_mvtorch.cache_write takes 9 arguments");
  const at::Tensor *slots = plain(a[0]), *k = plain(a[2]), *v = plain(a[3]), *kc = plain(a[4]), *vc = plain(a[5]),
                   *given = plain(a[6]);
  const int64_t total_slots = PyLong_AsLongLong(a[1]), bs = PyLong_AsLongLong(a[7]);
  if (PyErr_Occurred()) return nullptr;
  if (!slots || !k || !v || !kc || !vc || !given || k->dim() != 3 || !k->is_cuda() || k->sizes() != v->sizes() ||
      v->scalar_type() != k->scalar_type() || v->device() != k->device() || dtype_code(k->scalar_type()) < 0 ||
      !caches_ok(*kc, *vc, *k) || kc->size(1) != k->size(1) || kc->size(3) != k->size(2) || kc->size(2) != bs ||
      kc->size(0) * bs != total_slots || slots->device() != k->device() || slots->scalar_type() != at::kLong ||
      !slots->is_contiguous() || !sized(*given, {k->size(0)}) || !sized(*slots, {k->size(0)}) || k->size(0) == 0 ||
      k->stride(2) != 1 || v->stride(2) != 1)
    return none();
  const int rc = g_cache_write(k->data_ptr(), k->stride(0), k->stride(1), v->data_ptr(), v->stride(0), v->stride(1),
                               kc->data_ptr(), vc->data_ptr(), slots->data_ptr<int64_t>(), k->size(0),
                               static_cast<int32_t>(k->size(1)), static_cast<int32_t>(k->size(2)),
                               static_cast<int32_t>(bs), kc->size(0), dtype_code(k->scalar_type()), address(a[8]));
  if (rc) return status(rc);
  Py_RETURN_TRUE;
  END_HANDLE_TH_ERRORS
}

// rope_write(checked slots, checked positions, total slots, table rows they
// were checked for, query, key, value, positions, cos, sin, key_cache,
// value_cache, slot_mapping, block_size, return_key, stream): (query out, key
// out or None)
PyObject* rope_write(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 16) return PyErr_Format(PyExc_TypeError, "_mvtorch.rope_write takes 16 arguments");
  const at::Tensor *slots = plain(a[0]), *pos = plain(a[1]), *q = plain(a[4]), *k = plain(a[5]), *v = plain(a[6]),
                   *pos_given = plain(a[7]), *cos = plain(a[8]), *sin = plain(a[9]), *kc = plain(a[10]),
                   *vc = plain(a[11]), *slots_given = plain(a[12]);
  const int64_t total_slots = PyLong_AsLongLong(a[2]), max_pos = PyLong_AsLongLong(a[3]);
  const int64_t bs = PyLong_AsLongLong(a[13]);
  const int return_key = PyObject_IsTrue(a[14]);
  if (PyErr_Occurred()) return nullptr;
  if (!slots || !pos || !q || !k || !v || !pos_given || !cos || !sin || !kc || !vc || !slots_given || q->dim() != 3 ||
      k->dim() != 3 || !k->is_cuda() || cos->dim() != 2)
    return none();
  const int64_t t = k->size(0), hkv = k->size(1), d = k->size(2);
  const auto like = [&](const at::Tensor& x) {
    return x.scalar_type() == k->scalar_type() && x.device() == k->device();
  };
  Rows rq, rk, rv;
  if (t == 0 || dtype_code(k->scalar_type()) < 0 || !like(*q) || !like(*v) || !like(*cos) || !like(*sin) ||
      q->size(0) != t || q->size(2) != d || k->sizes() != v->sizes() || cos->sizes() != sin->sizes() ||
      cos->size(0) != max_pos || cos->size(1) < d || cos->stride(1) != 1 || sin->stride(1) != 1 ||
      cos->stride(0) != sin->stride(0) || !caches_ok(*kc, *vc, *k) || kc->size(1) != hkv || kc->size(3) != d ||
      kc->size(2) != bs || kc->size(0) * bs != total_slots || (bs & (bs - 1)) || !sized(*slots, {t}) ||
      !sized(*pos, {t}) || !sized(*pos_given, {t}) || !sized(*slots_given, {t}) || slots->device() != k->device() ||
      pos->device() != k->device() || slots->scalar_type() != at::kLong || pos->scalar_type() != at::kLong ||
      !slots->is_contiguous() || !pos->is_contiguous() || !aligned_rows(*q, rq) || !aligned_rows(*k, rk) ||
      !aligned_rows(*v, rv))
    return none();
  at::Tensor q_out = at::empty(q->sizes(), q->options()), k_out;
  if (return_key) k_out = at::empty(k->sizes(), k->options());
  const int64_t hq = q->size(1);
  const int rc = g_rope_write(
      rq.p, rq.st, rq.sh, q_out.data_ptr(), hq * d, d, rk.p, rk.st, rk.sh, return_key ? k_out.data_ptr() : nullptr,
      return_key ? hkv * d : 0, return_key ? d : 0, rv.p, rv.st, rv.sh, kc->data_ptr(), vc->data_ptr(),
      slots->data_ptr<int64_t>(), pos->data_ptr<int64_t>(), cos->data_ptr(), sin->data_ptr(), cos->stride(0), max_pos,
      t, static_cast<int32_t>(hq), static_cast<int32_t>(hkv), static_cast<int32_t>(d), static_cast<int32_t>(bs),
      kc->size(0), dtype_code(k->scalar_type()), address(a[15]));
  if (rc) return status(rc);
  PyObject* qo = THPVariable_Wrap(std::move(q_out));
  PyObject* ko = return_key ? THPVariable_Wrap(std::move(k_out)) : Py_NewRef(Py_None);
  PyObject* pair = qo && ko ? PyTuple_Pack(2, qo, ko) : nullptr;
  Py_XDECREF(qo);
  Py_XDECREF(ko);
  return pair;
  END_HANDLE_TH_ERRORS
}

// prefill(plan words, query, key, value, key_cache, value_cache, rows of out, stream)
PyObject* prefill(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 8) return PyErr_Format(PyExc_TypeError, "_mvtorch.prefill takes 8 arguments");
  const Words w(a[0], 20);
  const at::Tensor *q = plain(a[1]), *k = plain(a[2]), *v = plain(a[3]), *kc = plain(a[4]), *vc = plain(a[5]);
  const int64_t rows = PyLong_AsLongLong(a[6]);
  if (PyErr_Occurred()) return nullptr;
  if (!w.p || !q || !k || !v || !kc || !vc || q->dim() != 3 || k->dim() != 3 || !q->is_cuda()) return none();
  const int64_t hq = w.i(11), hkv = w.i(12), d = w.i(13), bs = w.i(14), nb = w.i(15);
  Rows rq, rk, rv;
  if (q->size(0) < rows || rows == 0 || q->size(1) != hq || q->size(2) != d || k->sizes() != v->sizes() ||
      k->size(0) < rows || k->size(1) != hkv || k->size(2) != d || dtype_code(q->scalar_type()) != w.i(16) ||
      k->scalar_type() != q->scalar_type() || v->scalar_type() != q->scalar_type() || k->device() != q->device() ||
      v->device() != q->device() || q->device().index() != w.i(19) || !caches_ok(*kc, *vc, *q) ||
      !sized(*kc, {nb, hkv, bs, d}) || !aligned_rows(*q, rq) || !aligned_rows(*k, rk) || !aligned_rows(*v, rv))
    return none();
  at::Tensor out = at::empty({rows, hq, d}, q->options());
  const int rc = g_prefill(
      rq.p, rq.st, rq.sh, rk.p, rk.st, rk.sh, rv.p, rv.st, rv.sh, kc->data_ptr(), vc->data_ptr(), w.ptr<const void>(0),
      static_cast<int32_t>(w.i(1)), w.i(2), w.ptr<const int64_t>(3), static_cast<int32_t>(w.i(4)),
      w.ptr<const int32_t>(5), static_cast<int32_t>(w.i(6)), static_cast<int32_t>(w.i(7)),
      static_cast<int32_t>(w.i(8)), static_cast<int32_t>(w.i(9)), out.data_ptr(), hq * d, d,
      static_cast<float>(w.f(10)), static_cast<int32_t>(hq), static_cast<int32_t>(hkv), static_cast<int32_t>(d),
      static_cast<int32_t>(bs), nb, static_cast<int32_t>(w.i(16)), w.ptr<void>(17), static_cast<size_t>(w.i(18)),
      address(a[7]));
  return rc ? status(rc) : THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// bind(decode_write, decode, cache_write, rope_write, prefill): the entry
// points' addresses in the loaded libmvattn.so.
PyObject* bind(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 5) return PyErr_Format(PyExc_TypeError, "_mvtorch.bind takes 5 addresses");
  void* p[5];
  for (int k = 0; k < 5; ++k) {
    p[k] = PyLong_AsVoidPtr(a[k]);
    if (PyErr_Occurred()) return nullptr;
    if (!p[k]) return PyErr_Format(PyExc_ValueError, "_mvtorch.bind: null address");
  }
  g_decode_write = reinterpret_cast<decltype(g_decode_write)>(p[0]);
  g_decode = reinterpret_cast<decltype(g_decode)>(p[1]);
  g_cache_write = reinterpret_cast<decltype(g_cache_write)>(p[2]);
  g_rope_write = reinterpret_cast<decltype(g_rope_write)>(p[3]);
  g_prefill = reinterpret_cast<decltype(g_prefill)>(p[4]);
  Py_RETURN_NONE;
}

#define FASTCALL(f) reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(f)), METH_FASTCALL
PyMethodDef methods[] = {
    {"bind", FASTCALL(bind), "bind the entry points"},
    {"seen", FASTCALL(seen), "weak references, versions, tensors: unchanged?"},
    {"decode_write", FASTCALL(decode_write), "mv_paged_decode_write of one layer of a step"},
    {"decode", FASTCALL(decode), "mv_paged_decode of one layer of a step"},
    {"cache_write", FASTCALL(cache_write), "mv_kv_cache_write of one layer of a step"},
    {"rope_write", FASTCALL(rope_write), "mv_rope_kv_cache_write of one layer of a step"},
    {"prefill", FASTCALL(prefill), "mv_paged_prefill_blocks of one layer of a step"},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_mvtorch", "per-layer launches of libmvattn", -1, methods,
                      nullptr, nullptr, nullptr, nullptr};

}  // namespace

// (ABI: the header this module was built against)
PyMODINIT_FUNC PyInit__mvtorch(void) {
  PyObject* m = PyModule_Create(&module);
  if (m && PyModule_AddIntConstant(m, "ABI", MVATTN_ABI_VERSION) < 0) {
    Py_DECREF(m);
    return nullptr;
  }
  return m;
}
