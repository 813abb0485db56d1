// Host side of the short calls, compiled: paged decode of a batch and the KV
// gather take microseconds on the device, and reading a dozen tensors'
// properties from Python took longer than that (5 x 1000 tokens, 8 x 96
// float32, two launches: 17.7 -> 9.4 us a call; 1 x 2048 bfloat16 with the
// append 18.9 -> 9.5 us; twelve layers of append and gather at 8192 tokens 188
// -> 152 us).  Each function here takes the tensors,
// checks the form the usual calls have, allocates the results and queues the
// launches through the library's C entry points; for any other form it returns
// None and the caller goes through the checks written in Python, which raise
// what is wrong.  A failed entry point's status is returned as an int.
#include <ATen/ATen.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <algorithm>
#include <cmath>
#include <vector>

#include "mie_paged_kv.h"

namespace {

// The entry points, from the library the process has already loaded.
decltype(&mie_paged_decode) g_decode;
decltype(&mie_paged_decode_append) g_decode_append;
decltype(&mie_paged_decode_plan) g_plan;
decltype(&mie_paged_decode_plan_known) g_plan_known;
decltype(&mie_kv_gather) g_gather;

// A plain ROCm tensor: no subclass, no functorch or dispatch wrapper, storage
// of its own device.
const at::Tensor* plain(PyObject* o) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  if (!t.is_cuda() || t.layout() != at::kStrided || t.is_neg() || t.is_conj()) return nullptr;
  const auto keys = t.key_set();
  if (keys.has_any(c10::DispatchKeySet({c10::DispatchKey::Python, c10::DispatchKey::FuncTorchBatched,
                                        c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::BatchedNestedTensor,
                                        c10::DispatchKey::Functionalize})))
    return nullptr;
  return &t;
}

int dtype_code(at::ScalarType t) {
  switch (t) {
    case at::kFloat: return MIE_DTYPE_F32;
    case at::kBFloat16: return MIE_DTYPE_BF16;
    default: return -1;
  }
}

bool as_int(PyObject* o, int64_t& out) {
  if (!PyLong_CheckExact(o)) return false;
  out = PyLong_AsLongLong(o);
  if (out == -1 && PyErr_Occurred()) {
    PyErr_Clear();
    return false;
  }
  return true;
}

bool fits(int64_t v) { return v >= 0 && v <= INT32_MAX; }

// decode(q, k_pool, v_pool, layer, tables, lens, max_len, host_lens, scale,
//        partition, k_new, v_new, stream) -> out, None or a status
// q [B, H, D], pools [L, NB, H, BS, D], tables int32 [B, n], lens int32 [B];
// host_lens a list of ints or None; scale a float or None; k_new, v_new
// [B, H, D] or None.
PyObject* decode(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 13) Py_RETURN_NONE;
  const at::Tensor *q = plain(a[0]), *k = plain(a[1]), *v = plain(a[2]), *tables = plain(a[4]), *lens = plain(a[5]);
  int64_t layer, max_len, partition, stream;
  if (!q || !k || !v || !tables || !lens || !as_int(a[3], layer) || !as_int(a[6], max_len) ||
      !as_int(a[9], partition) || !as_int(a[12], stream))
    Py_RETURN_NONE;
  if (q->dim() != 3 || k->dim() != 5 || tables->dim() != 2 || lens->dim() != 1) Py_RETURN_NONE;
  const auto qs = q->sizes(), ks = k->sizes();
  const auto qt = q->strides(), kt = k->strides();
  const int code = dtype_code(q->scalar_type());
  const auto device = q->device();
  const int64_t batch = qs[0], heads = qs[1], dim = qs[2], blocks = ks[1], block = ks[3];
  if (code < 0 || k->scalar_type() != q->scalar_type() || v->scalar_type() != q->scalar_type() ||
      k->device() != device || v->device() != device || tables->device() != device || lens->device() != device ||
      tables->scalar_type() != at::kInt || lens->scalar_type() != at::kInt || v->sizes() != ks || v->strides() != kt ||
      layer < 0 || layer >= ks[0] || ks[2] != heads || ks[4] != dim || kt[4] != 1 || kt[3] != dim || qt[2] != 1 ||
      tables->size(0) != batch || tables->stride(1) != 1 || lens->size(0) != batch || !lens->is_contiguous() ||
      !fits(batch) || !fits(heads) || !fits(blocks) || !fits(block) || !fits(max_len) || partition < -1 ||
      partition > INT32_MAX)
    Py_RETURN_NONE;
  double scale = 1.0 / std::sqrt(static_cast<double>(dim));
  if (a[8] != Py_None) {
    if (!PyFloat_CheckExact(a[8])) Py_RETURN_NONE;
    scale = PyFloat_AS_DOUBLE(a[8]);
  }
  std::vector<int32_t> host;
  int64_t longest = 0;
  if (a[7] != Py_None) {
    if (!PyList_CheckExact(a[7]) || PyList_GET_SIZE(a[7]) != batch) Py_RETURN_NONE;
    host.resize(batch);
    for (int64_t b = 0; b < batch; ++b) {
      int64_t c;
      if (!as_int(PyList_GET_ITEM(a[7], b), c) || c < INT32_MIN || c > INT32_MAX) Py_RETURN_NONE;
      host[b] = static_cast<int32_t>(c);
      longest = std::max(longest, std::min(c, max_len));
    }
  }
  const at::Tensor *kn = nullptr, *vn = nullptr;
  if (a[10] != Py_None || a[11] != Py_None) {
    kn = plain(a[10]);
    vn = plain(a[11]);
    for (const at::Tensor* t : {kn, vn})
      if (!t || t->sizes() != qs || t->scalar_type() != q->scalar_type() || t->device() != device || t->stride(2) != 1)
        Py_RETURN_NONE;
    if (kn->strides() != vn->strides()) Py_RETURN_NONE;
  }
  int32_t part = static_cast<int32_t>(partition);
  int64_t bytes = 0;
  int32_t rc = a[7] != Py_None && partition == 0
                   ? g_plan_known(batch, heads, dim, block, max_len, longest, kn != nullptr, code, &part, &bytes)
                   : g_plan(batch, heads, dim, block, max_len, code, partition, nullptr, &bytes);
  if (rc != MIE_OK) return PyLong_FromLong(rc);
  at::Tensor out = at::empty({batch, heads, dim}, q->options().requires_grad(false));
  at::Tensor ws;
  if (bytes > 0) ws = at::empty({bytes}, q->options().dtype(at::kByte).requires_grad(false));
  const int64_t offset = layer * kt[0] * q->element_size();
  char* kp = static_cast<char*>(k->data_ptr()) + offset;
  char* vp = static_cast<char*>(v->data_ptr()) + offset;
  const int32_t* tab = static_cast<const int32_t*>(tables->data_ptr());
  const int32_t* len = static_cast<const int32_t*>(lens->data_ptr());
  const int32_t* hl = host.empty() ? nullptr : host.data();
  void* wsp = bytes > 0 ? ws.data_ptr() : nullptr;
  void* st = reinterpret_cast<void*>(stream);
  void* op = out.data_ptr();
  const void* qp = q->data_ptr();
  const void* knp = kn ? kn->data_ptr() : nullptr;
  const void* vnp = vn ? vn->data_ptr() : nullptr;
  const int64_t nb = kn ? kn->stride(0) : 0, nh = kn ? kn->stride(1) : 0, ts = tables->stride(0);
  // A launch waits when the queue is full: not with the interpreter held.
  Py_BEGIN_ALLOW_THREADS
  if (kn) {
    rc = g_decode_append(qp, qt[0], qt[1], kp, vp, kt[1], kt[2], blocks, tab, ts, len, hl, 0, max_len, batch, heads,
                         dim, block, static_cast<float>(scale), op, heads * dim, dim, code, wsp, bytes, part, knp,
                         vnp, nb, nh, code, st);
  } else {
    rc = g_decode(qp, qt[0], qt[1], kp, vp, kt[1], kt[2], blocks, tab, ts, len, hl, 0, max_len, batch, heads, dim,
                  block, static_cast<float>(scale), op, heads * dim, dim, code, wsp, bytes, part, code, st);
  }
  Py_END_ALLOW_THREADS
  if (rc != MIE_OK) return PyLong_FromLong(rc);
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// gather(k_pool, v_pool, layer, table, length, stream) -> (K, V), None or a status
// Contiguous pools [L, NB, H, BS, D] of one dtype, table int32 with an entry
// per block of the pool.
PyObject* gather(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 6) Py_RETURN_NONE;
  const at::Tensor *k = plain(a[0]), *v = plain(a[1]), *table = plain(a[3]);
  int64_t layer, length, stream;
  if (!k || !v || !table || !as_int(a[2], layer) || !as_int(a[4], length) || !as_int(a[5], stream)) Py_RETURN_NONE;
  const int code = dtype_code(k->scalar_type());
  if (k->dim() != 5 || code < 0 || v->scalar_type() != k->scalar_type() || v->sizes() != k->sizes() ||
      !k->is_contiguous() || !v->is_contiguous() || v->device() != k->device() || table->device() != k->device() ||
      table->scalar_type() != at::kInt || table->dim() != 1 || !table->is_contiguous())
    Py_RETURN_NONE;
  const auto s = k->sizes();
  const int64_t blocks = s[1], heads = s[2], block = s[3], dim = s[4];
  if (layer < 0 || layer >= s[0] || !fits(blocks) || !fits(heads) || !fits(block) || !fits(dim) || !fits(length) ||
      length > blocks * block || table->size(0) < blocks)
    Py_RETURN_NONE;
  const auto options = k->options().requires_grad(false);
  at::Tensor ko = at::empty({1, heads, length, dim}, options), vo = at::empty({1, heads, length, dim}, options);
  const int64_t tile = block * dim, offset = layer * blocks * heads * tile * k->element_size();
  const char* kp = static_cast<const char*>(k->data_ptr()) + offset;
  const char* vp = static_cast<const char*>(v->data_ptr()) + offset;
  const int32_t* tab = static_cast<const int32_t*>(table->data_ptr());
  void *kop = ko.data_ptr(), *vop = vo.data_ptr();
  int32_t rc;
  Py_BEGIN_ALLOW_THREADS
  rc = g_gather(kp, vp, heads * tile, tile, blocks, tab, length, kop, vop, length * dim, dim, heads, dim, block, code,
                reinterpret_cast<void*>(stream));
  Py_END_ALLOW_THREADS
  if (rc != MIE_OK) return PyLong_FromLong(rc);
  PyObject* pair = PyTuple_New(2);
  if (!pair) return nullptr;
  PyTuple_SET_ITEM(pair, 0, THPVariable_Wrap(std::move(ko)));
  PyTuple_SET_ITEM(pair, 1, THPVariable_Wrap(std::move(vo)));
  return pair;
  END_HANDLE_TH_ERRORS
}

// bind(decode, decode_append, plan, plan_known, gather): the entry points' addresses.
PyObject* bind(PyObject*, PyObject* const* a, Py_ssize_t n) {
  void* p[5];
  if (n != 5) {
    PyErr_SetString(PyExc_TypeError, "bind takes five addresses");
    return nullptr;
  }
  for (int i = 0; i < 5; ++i) {
    p[i] = PyLong_AsVoidPtr(a[i]);
    if (!p[i]) {
      if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "bind: null address");
      return nullptr;
    }
  }
  g_decode = reinterpret_cast<decltype(g_decode)>(p[0]);
  g_decode_append = reinterpret_cast<decltype(g_decode_append)>(p[1]);
  g_plan = reinterpret_cast<decltype(g_plan)>(p[2]);
  g_plan_known = reinterpret_cast<decltype(g_plan_known)>(p[3]);
  g_gather = reinterpret_cast<decltype(g_gather)>(p[4]);
  Py_RETURN_NONE;
}

PyMethodDef g_methods[] = {
    {"decode", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(decode)), METH_FASTCALL, nullptr},
    {"gather", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(gather)), METH_FASTCALL, nullptr},
    {"bind", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(bind)), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_host_calls", nullptr, -1, g_methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

// abi_version: the header's version these calls were compiled for; bind() is
// for a library of the same one.
PyMODINIT_FUNC PyInit__host_calls() {
  PyObject* m = PyModule_Create(&g_module);
  if (m && PyModule_AddIntConstant(m, "abi_version", MIE_ABI_VERSION) < 0) {
    Py_DECREF(m);
    return nullptr;
  }
  return m;
}
