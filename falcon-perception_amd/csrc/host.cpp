// The calls an eager layer makes (append, decode step, prefill attention) from PyTorch tensors to the C ABI of
// include/fp_paged_kv.h, as a Python module.
//
// Bound by the host: a layer of a small eager step is shorter on the GPU than its calls are in Python, where every pointer, size
// and stride is an attribute look-up and the foreign call converts forty arguments one by one.  Here they are read from the tensors in C++:
// four short fp32 sequences, 28 layers, without graphs 818 -> 380 us a step (29 -> 13.5 us a layer, of which the GPU works 7), one prompt
// of 613 rows 911 -> 700 us (33 -> 25 us a layer, now the GPU's).
//
// The functions take the tensors as ops.py would hand them to the library.  What they do not recognise at once (a tensor
// subclass, another device or type, rows that are not dense, shapes that do not match) they leave alone and return None: ops.py
// then converts the arguments or says what is wrong with them.  Nothing is kept from one call to the next.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/version.h>

#include <exception>

#include "fp_paged_kv.h"

namespace {

// The tensor behind a Python object, or null: not a plain tensor on the GPU.
const at::Tensor* gpu_tensor(PyObject* o) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  return t.is_cuda() && t.layout() == at::kStrided ? &t : nullptr;
}

int dtype_code(const at::Tensor& t) {
  switch (t.scalar_type()) {
    case at::kFloat: return FP_DTYPE_F32;
    case at::kBFloat16: return FP_DTYPE_BF16;
    case at::kHalf: return FP_DTYPE_F16;
    default: return -1;
  }
}

int index_code(const at::Tensor& t) {
  return t.scalar_type() == at::kInt ? FP_INDEX_I32 : t.scalar_type() == at::kLong ? FP_INDEX_I64 : -1;
}

bool is_table(const at::Tensor& t) { return t.dim() == 2 && t.scalar_type() == at::kLong && t.stride(1) == 1; }
bool is_indices(const at::Tensor& t, int64_t n) { return t.scalar_type() == at::kLong && t.is_contiguous() && t.numel() == n; }
bool is_bytes(const at::Tensor& t) { return t.scalar_type() == at::kByte && t.is_contiguous(); }
bool dense_rows(const at::Tensor& t) { return t.stride(t.dim() - 1) == 1; }

// Other Python threads run while this one allocates and launches, which may wait (for a full queue, or for memory).
struct Unlocked {
  PyThreadState* const thread = PyEval_SaveThread();
  Unlocked() = default;
  Unlocked(const Unlocked&) = delete;
  ~Unlocked() { PyEval_RestoreThread(thread); }
};

PyObject* fail(const char* what, int rc) {
  PyErr_Format(PyExc_RuntimeError, "%s failed (%d): %s", what, rc, fp_last_error());
  return nullptr;
}

// One call's arguments, taken in order.  `ok` turns false at the first that is not what was asked for.
struct Args {
  PyObject* const* at;
  bool ok = true;
  const at::Tensor* tensor() {
    const at::Tensor* t = gpu_tensor(*at++);
    if (!t) ok = false;
    return t;
  }
  const at::Tensor* maybe_tensor() {  // null for None
    if (*at == Py_None) {
      ++at;
      return nullptr;
    }
    return tensor();
  }
  int64_t integer() {
    const long long v = PyLong_AsLongLong(*at++);
    if (v == -1 && PyErr_Occurred()) {
      PyErr_Clear();
      ok = false;
    }
    return v;
  }
  double number() {
    const double v = PyFloat_AsDouble(*at++);
    if (v == -1.0 && PyErr_Occurred()) {
      PyErr_Clear();
      ok = false;
    }
    return v;
  }
};

PyObject* pair(const at::Tensor& a, const at::Tensor& b) {
  PyObject* t = PyTuple_New(2);
  if (!t) return nullptr;
  PyTuple_SET_ITEM(t, 0, THPVariable_Wrap(a));
  PyTuple_SET_ITEM(t, 1, THPVariable_Wrap(b));
  return t;
}

// pool_k, pool_v, k, v, page_table, batch_idx, input_pos, page_size, clamp_negative, packed, stream -> True
PyObject* append_unguarded(PyObject* const* args) {
  Args a{args};
  const at::Tensor *pk = a.tensor(), *pv = a.tensor(), *k = a.tensor(), *v = a.tensor(), *table = a.tensor(), *bidx = a.tensor(),
                   *pos = a.tensor();
  const int64_t page_size = a.integer(), clamp = a.integer(), packed = a.integer(), stream = a.integer();
  if (!a.ok) Py_RETURN_NONE;
  const int dt = dtype_code(*k), it = index_code(*pos);
  if (dt < 0 || it < 0 || k->dim() != 4 || k->sizes() != v->sizes() || v->scalar_type() != k->scalar_type() ||
      pk->scalar_type() != k->scalar_type() || pv->scalar_type() != k->scalar_type() || pk->dim() != 3 || !pk->is_contiguous() ||
      !pv->is_contiguous() || !dense_rows(*k) || !dense_rows(*v) || !is_table(*table) || !pos->is_contiguous())
    Py_RETURN_NONE;
  int64_t T, H, S, ks[3], vs[3];
  const int64_t D = k->size(3);
  if (packed) {
    T = k->size(2), H = k->size(1), S = 1;
    if (k->size(0) != 1 || pos->numel() != T) Py_RETURN_NONE;
    ks[0] = k->stride(2), ks[1] = k->stride(1), ks[2] = 0;
    vs[0] = v->stride(2), vs[1] = v->stride(1), vs[2] = 0;
  } else {
    T = k->size(0), H = k->size(1), S = k->size(2);
    if (pos->numel() != T * S) Py_RETURN_NONE;
    for (int i = 0; i < 3; ++i) ks[i] = k->stride(i), vs[i] = v->stride(i);
  }
  if (!is_indices(*bidx, T)) Py_RETURN_NONE;
  int rc;
  {
    const Unlocked others;
    rc = fp_kv_append(pk->data_ptr(), pv->data_ptr(), k->data_ptr(), v->data_ptr(), ks[0], ks[1], ks[2], vs[0], vs[1], vs[2],
                      static_cast<const int64_t*>(table->data_ptr()), table->stride(0),
                      static_cast<const int64_t*>(bidx->data_ptr()), pos->data_ptr(), it, T, H, S, D, page_size,
                      table->size(1), table->size(0), pk->size(1), dt, clamp ? 1 : 0, reinterpret_cast<void*>(stream));
  }
  if (rc < 0) return fail("fp_kv_append", rc);
  Py_RETURN_TRUE;
}

// q, pool_k, pool_v, page_table, batch_idx, input_pos, page_size, max_context, scale, split_tokens, workspace, sinks, kv_rep,
// k_new, v_new, plan, arrivals, next_arrivals, stream -> (out, lse)
PyObject* decode_unguarded(PyObject* const* args) {
  Args a{args};
  const at::Tensor *q = a.tensor(), *pk = a.tensor(), *pv = a.tensor(), *table = a.tensor(), *bidx = a.tensor(), *pos = a.tensor();
  const int64_t page_size = a.integer(), max_context = a.integer();
  const double scale = a.number();
  const int64_t split_tokens = a.integer();
  const at::Tensor *ws = a.maybe_tensor(), *sinks = a.maybe_tensor();
  const int64_t kv_rep = a.integer();
  const at::Tensor *kn = a.maybe_tensor(), *vn = a.maybe_tensor(), *plan = a.maybe_tensor(), *arrivals = a.tensor(),
                   *after = a.maybe_tensor();
  const int64_t stream = a.integer();
  if (!a.ok) Py_RETURN_NONE;
  const int dt = dtype_code(*q), it = index_code(*pos);
  if (dt < 0 || it < 0 || q->dim() != 4 || q->size(2) != 1 || pk->dim() != 3 || pk->sizes() != pv->sizes() ||
      pk->size(2) != q->size(3) || pk->scalar_type() != q->scalar_type() || pv->scalar_type() != q->scalar_type() ||
      !pk->is_contiguous() || !pv->is_contiguous() || !dense_rows(*q) || !is_table(*table) || split_tokens <= 0 || kv_rep < 1)
    Py_RETURN_NONE;
  const int64_t B = q->size(0), Hq = q->size(1), D = q->size(3), Hc = pk->size(0);
  if (!is_indices(*bidx, B) || pos->numel() != B || !pos->is_contiguous() || (ws && !is_bytes(*ws)) || (plan && !is_bytes(*plan)) ||
      arrivals->scalar_type() != at::kInt || !arrivals->is_contiguous() ||
      (after && (after->scalar_type() != at::kInt || !after->is_contiguous() || after->numel() != arrivals->numel())) ||
      (sinks && (sinks->scalar_type() != at::kFloat || sinks->dim() != 1 || sinks->size(0) != Hq || !sinks->is_contiguous() ||
                 sinks->device() != q->device())))
    Py_RETURN_NONE;
  if (!kn != !vn) Py_RETURN_NONE;
  if (kn) {
    const int64_t fresh[4] = {B, Hc, 1, D};
    if (kn->sizes() != at::IntArrayRef(fresh, 4) || vn->sizes() != at::IntArrayRef(fresh, 4) || kn->scalar_type() != q->scalar_type() ||
        vn->scalar_type() != q->scalar_type() || !dense_rows(*kn) || !dense_rows(*vn))
      Py_RETURN_NONE;
  }
  at::Tensor out, lse;
  int rc;
  {
    const Unlocked others;
    out = at::empty({B, Hq, 1, D}, q->options());
    lse = at::empty({B, Hq, 1}, q->options().dtype(at::kFloat));
    rc = fp_paged_decode_step(
        static_cast<int32_t*>(arrivals->data_ptr()), after ? static_cast<int32_t*>(after->data_ptr()) : nullptr,
        arrivals->numel() * 4, kn ? kn->data_ptr() : nullptr, vn ? vn->data_ptr() : nullptr,
        kn ? kn->stride(0) : 0, kn ? kn->stride(1) : 0, vn ? vn->stride(0) : 0, vn ? vn->stride(1) : 0, q->data_ptr(), q->stride(0),
        q->stride(1), pk->data_ptr(), pv->data_ptr(), static_cast<const int64_t*>(table->data_ptr()), table->stride(0),
        static_cast<const int64_t*>(bidx->data_ptr()), pos->data_ptr(), it, out.data_ptr(), out.stride(0), out.stride(1),
        static_cast<float*>(lse.data_ptr()), sinks ? static_cast<const float*>(sinks->data_ptr()) : nullptr, ws ? ws->data_ptr() : nullptr,
        ws ? ws->numel() : 0, B, Hq, Hc, kv_rep, D, page_size, table->size(1), table->size(0), pk->size(1), max_context, split_tokens,
        static_cast<float>(scale), dt, plan ? plan->data_ptr() : nullptr, plan ? plan->numel() : 0, reinterpret_cast<void*>(stream));
  }
  if (rc < 0) return fail("fp_paged_decode_step", rc);
  return pair(out, lse);
}

// q, pool_k, pool_v, page_table, batch_idx, row_limit, page_size, scale, sinks, workspace, score_bound, tile_order, order_rows,
// stream -> (out, lse)
PyObject* prefill_unguarded(PyObject* const* args) {
  Args a{args};
  const at::Tensor *q = a.tensor(), *pk = a.tensor(), *pv = a.tensor(), *table = a.tensor(), *bidx = a.tensor(), *limit = a.tensor();
  const int64_t page_size = a.integer();
  const double scale = a.number();
  const at::Tensor *sinks = a.maybe_tensor(), *ws = a.maybe_tensor();
  const double bound = a.number();
  const at::Tensor* order = a.maybe_tensor();
  const int64_t order_rows = a.integer(), stream = a.integer();
  if (!a.ok) Py_RETURN_NONE;
  const int dt = dtype_code(*q);
  if (dt < 0 || q->dim() != 4 || q->size(0) != 1 || pk->dim() != 3 || pk->sizes() != pv->sizes() || pk->size(2) != q->size(3) ||
      pk->scalar_type() != q->scalar_type() || pv->scalar_type() != q->scalar_type() || !pk->is_contiguous() || !pv->is_contiguous() ||
      !dense_rows(*q) || !is_table(*table))
    Py_RETURN_NONE;
  const int64_t Hq = q->size(1), Lq = q->size(2), D = q->size(3), Hc = pk->size(0);
  if (!is_indices(*bidx, Lq) || limit->scalar_type() != at::kInt || !limit->is_contiguous() || limit->numel() != Lq ||
      (ws && !is_bytes(*ws)) ||
      (sinks && (sinks->scalar_type() != at::kFloat || sinks->dim() != 1 || sinks->size(0) != Hq || !sinks->is_contiguous() ||
                 sinks->device() != q->device())) ||
      (order && (order_rows <= 0 || order->scalar_type() != at::kInt || !order->is_contiguous() ||
                 order->numel() != (Lq + order_rows - 1) / order_rows)))
    Py_RETURN_NONE;
  at::Tensor out, lse;
  int rc = FP_OK;
  {
    const Unlocked others;
    out = at::empty_like(*q);
    lse = at::empty({1, Hq, Lq}, q->options().dtype(at::kFloat));
    if (dense_rows(out))
      rc = fp_paged_prefill(
          q->data_ptr(), q->stride(2), q->stride(1), pk->data_ptr(), pv->data_ptr(), static_cast<const int64_t*>(table->data_ptr()),
          table->stride(0), static_cast<const int64_t*>(bidx->data_ptr()), static_cast<const int32_t*>(limit->data_ptr()), out.data_ptr(),
          out.stride(2), out.stride(1), static_cast<float*>(lse.data_ptr()), sinks ? static_cast<const float*>(sinks->data_ptr()) : nullptr,
          Lq, Hq, Hc, D, page_size, table->size(1), table->size(0), pk->size(1), static_cast<float>(scale), static_cast<float>(bound), dt,
          ws ? ws->data_ptr() : nullptr, ws ? ws->numel() : 0, order ? static_cast<const int32_t*>(order->data_ptr()) : nullptr,
          order ? order_rows : 0, reinterpret_cast<void*>(stream));
  }
  if (!dense_rows(out)) Py_RETURN_NONE;
  if (rc < 0) return fail("fp_paged_prefill", rc);
  return pair(out, lse);
}

// A C++ exception (an allocation that failed) becomes a Python one.
template <PyObject* (*kCall)(PyObject* const*), Py_ssize_t kArgs>
PyObject* guarded(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (n != kArgs) {
    PyErr_Format(PyExc_TypeError, "%zd arguments expected, %zd given", kArgs, n);
    return nullptr;
  }
  HANDLE_TH_ERRORS
  return kCall(args);
  END_HANDLE_TH_ERRORS
}

#define FP_METHOD(name, call, n) {name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(guarded<call, n>)), METH_FASTCALL, nullptr}
PyMethodDef kMethods[] = {FP_METHOD("append", append_unguarded, 11), FP_METHOD("decode", decode_unguarded, 19),
                          FP_METHOD("prefill", prefill_unguarded, 14), {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "fp_host", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_fp_host() {
  if (fp_abi_version() != FP_ABI_VERSION) {
    PyErr_Format(PyExc_RuntimeError, "libfp_paged_kv.so has ABI %d, fp_host was built for %d", fp_abi_version(), FP_ABI_VERSION);
    return nullptr;
  }
  PyObject* const module = PyModule_Create(&kModule);
  if (module) PyModule_AddStringConstant(module, "torch_version", TORCH_VERSION);
  return module;
}
