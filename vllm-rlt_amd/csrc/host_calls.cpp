// Host side of the hot entry points: one C++ call from Python tensors to the C
// ABI.
//
// Checking a decode call's tensors, building its 29 C arguments and allocating
// its result in Python took 11 us of a 15 us call, twice what the kernel of a
// small batch runs.  The functions here do the same for the calls a serving
// loop makes: plain dense device tensors that pass every check.  Anything else
// (a failed check, a tensor subclass, an active function or dispatch mode, an
// empty batch) returns None before anything was done, and the caller takes
// the Python path, which raises the errors and handles the rest.  They return
// the result tensor, or the library's status when the launch was refused.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/TensorSubclassLikeUtils.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cmath>
#include <cstdint>

#include "rlt_kv.h"

namespace {

// Entry points of the library the Python package loaded (set by bind()).
decltype(&rlt_paged_decode) g_decode = nullptr;
decltype(&rlt_paged_decode_append) g_decode_append = nullptr;
decltype(&rlt_paged_decode_workspace_bytes) g_decode_bytes = nullptr;
decltype(&rlt_paged_prefill_split) g_prefill = nullptr;
decltype(&rlt_paged_prefill_split_workspace_bytes) g_prefill_bytes = nullptr;
decltype(&rlt_rope_kv_append) g_rope = nullptr;

// A plain device tensor of torch.Tensor itself, or null.  (Parameters and other
// subclasses, wrappers of vmap / grad and fake tensors take the Python path.)
const at::Tensor* plain(PyObject* o) {
  if (Py_TYPE(o) != reinterpret_cast<PyTypeObject*>(THPVariableClass)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || at::isTensorSubclassLike(t)) return nullptr;
  return &t;
}

bool modes_active() {
  return at::impl::torch_function_mode_enabled() || c10::impl::TorchDispatchModeTLS::any_modes_set();
}

int code_of(at::ScalarType t) {
  switch (t) {
    case at::kFloat: return RLT_FLOAT32;
    case at::kHalf: return RLT_FLOAT16;
    case at::kBFloat16: return RLT_BFLOAT16;
    default: return -1;
  }
}

bool aligned_rows(const at::Tensor& t) {
  if (t.stride(-1) != 1 || reinterpret_cast<uintptr_t>(t.data_ptr()) % 16) return false;
  for (int64_t i = 0; i + 1 < t.dim(); ++i)
    if (t.stride(i) * t.element_size() % 16) return false;
  return true;
}

bool ints(const at::Tensor& t, at::ScalarType type) {
  return t.scalar_type() == type && t.dim() == 1 && t.is_contiguous();
}

// Layer-slice caches and q of one dtype and device: [blocks, page, kv heads, d]
// and [rows, heads, d].
bool attention_shapes(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, const at::Tensor& tables,
                      const at::Tensor& lens) {
  return q.dim() == 3 && k.dim() == 4 && k.sizes() == v.sizes() && k.strides() == v.strides() &&
         q.size(2) == k.size(3) && k.size(2) > 0 && q.size(1) > 0 && q.size(1) % k.size(2) == 0 &&
         code_of(q.scalar_type()) >= 0 && k.scalar_type() == q.scalar_type() && v.scalar_type() == q.scalar_type() &&
         tables.scalar_type() == at::kInt && tables.dim() == 2 && tables.stride(1) == 1 && ints(lens, at::kInt) &&
         k.device() == q.device() && v.device() == q.device() && tables.device() == q.device() &&
         lens.device() == q.device();
}

// out when given and fitting (checked), a new tensor like q for None.
bool result_like(PyObject* o, const at::Tensor& q, at::Tensor* out) {
  if (o == Py_None) {
    *out = at::empty_like(q);
    return true;
  }
  const at::Tensor* t = plain(o);
  if (!t || t->sizes() != q.sizes() || t->scalar_type() != q.scalar_type() || t->device() != q.device()) return false;
  *out = *t;
  return true;
}

float scale_of(PyObject* o, int64_t d) {
  return static_cast<float>(o == Py_None ? 1.0 / std::sqrt(static_cast<double>(d)) : PyFloat_AS_DOUBLE(o));
}
bool scale_ok(PyObject* o) { return o == Py_None || PyFloat_CheckExact(o); }

PyObject* result(int rc, const at::Tensor& out) {
  if (rc != RLT_OK) return PyLong_FromLong(rc);
  return THPVariable_Wrap(out);
}

// decode(q, key, value, tables, lengths, out, workspace, scale, stream,
//        k_new, v_new, write_blocks, write_offsets, n_write); the last five
// absent for a decode without append, n_write None for all of write_blocks.
PyObject* decode(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  if ((nargs != 9 && nargs != 14) || modes_active()) Py_RETURN_NONE;
  const at::Tensor* in[5];
  for (int i = 0; i < 5; ++i)
    if (!(in[i] = plain(args[i]))) Py_RETURN_NONE;
  const at::Tensor &q = *in[0], &k = *in[1], &v = *in[2], &tables = *in[3], &lens = *in[4];
  if (!attention_shapes(q, k, v, tables, lens) || !scale_ok(args[7]) || !PyLong_CheckExact(args[8])) Py_RETURN_NONE;
  const int64_t rows = q.size(0), hq = q.size(1), d = q.size(2), hkv = k.size(2);
  if (rows == 0 || tables.size(0) != rows || lens.size(0) != rows) Py_RETURN_NONE;
  const at::Tensor* app[4] = {};
  int64_t n = 0;
  if (nargs == 14) {
    for (int i = 0; i < 4; ++i)
      if (!(app[i] = plain(args[9 + i])) || app[i]->device() != q.device()) Py_RETURN_NONE;
    if (!ints(*app[2], at::kLong) || !ints(*app[3], at::kLong)) Py_RETURN_NONE;
    if (args[13] == Py_None) n = app[2]->size(0);
    else if (PyLong_CheckExact(args[13])) n = PyLong_AsLongLong(args[13]);
    else Py_RETURN_NONE;
    if (PyErr_Occurred()) {  // n_write past 64 bits
      PyErr_Clear();
      Py_RETURN_NONE;
    }
    if (n < 0 || n > rows || n > app[2]->size(0) || n > app[3]->size(0)) Py_RETURN_NONE;
    for (int i = 0; i < 2; ++i)
      if (app[i]->dim() != 3 || app[i]->size(1) != hkv || app[i]->size(2) != d || app[i]->size(0) < n ||
          app[i]->scalar_type() != q.scalar_type())
        Py_RETURN_NONE;
  }
  const int64_t need = g_decode_bytes(rows, hq, hkv, d);
  at::Tensor workspace, out;
  if (args[6] != Py_None) {
    const at::Tensor* w = plain(args[6]);
    if (!w || w->device() != q.device() || w->numel() * static_cast<int64_t>(w->element_size()) < need) Py_RETURN_NONE;
    workspace = *w;
  }
  if (!result_like(args[5], q, &out)) Py_RETURN_NONE;
  if (!workspace.defined()) workspace = at::empty({need}, q.options().dtype(at::kByte));
  void* const stream = PyLong_AsVoidPtr(args[8]);
  const int64_t nbytes = workspace.numel() * static_cast<int64_t>(workspace.element_size());
  const float scale = scale_of(args[7], d);
  const int code = code_of(q.scalar_type());
  int rc;
  Py_BEGIN_ALLOW_THREADS  // as ctypes does
  if (nargs == 14) {
    rc = g_decode_append(q.data_ptr(), q.strides().data(), k.data_ptr(), v.data_ptr(), k.strides().data(),
                         tables.data_ptr<int32_t>(), tables.stride(0), tables.size(1), lens.data_ptr<int32_t>(),
                         out.data_ptr(), out.strides().data(), rows, hq, hkv, d, k.size(1), k.size(0), scale, code,
                         app[0]->data_ptr(), app[0]->strides().data(), app[1]->data_ptr(), app[1]->strides().data(),
                         app[2]->data_ptr<int64_t>(), app[3]->data_ptr<int64_t>(), n, workspace.data_ptr(), nbytes,
                         stream);
  } else {
    rc = g_decode(q.data_ptr(), q.strides().data(), k.data_ptr(), v.data_ptr(), k.strides().data(),
                  tables.data_ptr<int32_t>(), tables.stride(0), tables.size(1), lens.data_ptr<int32_t>(),
                  out.data_ptr(), out.strides().data(), rows, hq, hkv, d, k.size(1), k.size(0), scale, code,
                  workspace.data_ptr(), nbytes, stream);
  }
  Py_END_ALLOW_THREADS
  return result(rc, out);
  END_HANDLE_TH_ERRORS
}

// Workspace bytes of a prefill; rows off 16 bytes take the per-token path, whose
// workspace is the fp32 one's.
int64_t prefill_need(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, const at::Tensor& tables,
                     const at::Tensor& out) {
  const bool rows16 = aligned_rows(q) && aligned_rows(out) && aligned_rows(k) && aligned_rows(v);
  return g_prefill_bytes(q.size(0), tables.size(0), tables.size(1), q.size(1), k.size(2), q.size(2), k.size(1),
                         rows16 ? code_of(q.scalar_type()) : int{RLT_FLOAT32});
}

// prefill_bytes(q, key, value, tables): what prefill() needs of a given workspace.
PyObject* prefill_bytes(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  if (nargs != 4 || modes_active()) Py_RETURN_NONE;
  const at::Tensor* in[4];
  for (int i = 0; i < 4; ++i)
    if (!(in[i] = plain(args[i]))) Py_RETURN_NONE;
  const at::Tensor &q = *in[0], &k = *in[1], &v = *in[2], &tables = *in[3];
  if (q.dim() != 3 || k.dim() != 4 || v.dim() != 4 || tables.dim() != 2 || code_of(q.scalar_type()) < 0) Py_RETURN_NONE;
  return PyLong_FromLongLong(prefill_need(q, k, v, tables, q));
  END_HANDLE_TH_ERRORS
}

// prefill(q, key, value, tables, lengths, cu, max_seqlen_q, out, scale, stream,
//         workspace): the workspace for key segments or the per-token path is the
// given one when it is large enough, allocated here for None.
PyObject* prefill(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  if (nargs != 11 || modes_active()) Py_RETURN_NONE;
  const at::Tensor* in[6];
  for (int i = 0; i < 6; ++i)
    if (!(in[i] = plain(args[i]))) Py_RETURN_NONE;
  const at::Tensor &q = *in[0], &k = *in[1], &v = *in[2], &tables = *in[3], &lens = *in[4], &cu = *in[5];
  if (!attention_shapes(q, k, v, tables, lens) || !ints(cu, at::kInt) || cu.device() != q.device() ||
      !PyLong_CheckExact(args[6]) || !scale_ok(args[8]) || !PyLong_CheckExact(args[9]))
    Py_RETURN_NONE;
  const int64_t total = q.size(0), hq = q.size(1), d = q.size(2), hkv = k.size(2), nseq = tables.size(0);
  if (total == 0 || nseq == 0 || lens.size(0) != nseq || cu.size(0) != nseq + 1) Py_RETURN_NONE;
  const int64_t max_q = PyLong_AsLongLong(args[6]);
  if (max_q == -1 && PyErr_Occurred()) {
    PyErr_Clear();
    Py_RETURN_NONE;
  }
  at::Tensor out;
  if (!result_like(args[7], q, &out)) Py_RETURN_NONE;
  const int code = code_of(q.scalar_type());
  const int64_t need = prefill_need(q, k, v, tables, out);
  at::Tensor workspace;
  if (args[10] != Py_None) {
    const at::Tensor* w = plain(args[10]);
    if (!w || w->scalar_type() != at::kByte || w->device() != q.device() || w->numel() < need) Py_RETURN_NONE;
    workspace = *w;
  } else {
    workspace = at::empty({need > 0 ? need : 1}, q.options().dtype(at::kByte));
  }
  void* const stream = PyLong_AsVoidPtr(args[9]);
  const float scale = scale_of(args[8], d);
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = g_prefill(q.data_ptr(), q.strides().data(), k.data_ptr(), v.data_ptr(), k.strides().data(),
                 tables.data_ptr<int32_t>(), tables.stride(0), tables.size(1), lens.data_ptr<int32_t>(),
                 cu.data_ptr<int32_t>(), nseq, total, max_q, out.data_ptr(), out.strides().data(), hq, hkv, d, k.size(1),
                 k.size(0), scale, code, workspace.data_ptr(), workspace.numel(), stream);
  Py_END_ALLOW_THREADS
  return result(rc, out);
  END_HANDLE_TH_ERRORS
}

// rope(key_cache, value_cache, layer, write_blocks, write_offsets, q, k, v, cos,
//      sin, out, n_rows, stream); cos and sin [rows, d].
PyObject* rope(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  if (nargs != 13 || modes_active() || !PyLong_CheckExact(args[2]) || !PyLong_CheckExact(args[12])) Py_RETURN_NONE;
  static constexpr int kAt[9] = {0, 1, 3, 4, 5, 6, 7, 8, 9};
  const at::Tensor* in[9];
  for (int i = 0; i < 9; ++i)
    if (!(in[i] = plain(args[kAt[i]])) || in[i]->device() != in[0]->device()) Py_RETURN_NONE;
  const at::Tensor &kc = *in[0], &vc = *in[1], &wb = *in[2], &wo = *in[3], &q = *in[4], &k = *in[5], &v = *in[6],
                   &cos = *in[7], &sin = *in[8];
  if (kc.dim() != 5 || kc.sizes() != vc.sizes() || kc.strides() != vc.strides() || q.dim() != 3) Py_RETURN_NONE;
  const int64_t hkv = kc.size(3), d = kc.size(4), rows = q.size(0);
  const int code = code_of(kc.scalar_type());
  if (code < 0 || hkv == 0 || d % 2 || q.size(2) != d || q.size(1) % hkv || !ints(wb, at::kLong) || !ints(wo, at::kLong))
    Py_RETURN_NONE;
  for (const at::Tensor* t : {&k, &v})
    if (t->dim() != 3 || t->size(0) != rows || t->size(1) != hkv || t->size(2) != d) Py_RETURN_NONE;
  for (const at::Tensor* t : {&cos, &sin})
    if (t->dim() != 2 || t->size(0) != rows || t->size(1) != d) Py_RETURN_NONE;
  for (const at::Tensor* t : {&vc, &q, &k, &v, &cos, &sin})
    if (t->scalar_type() != kc.scalar_type()) Py_RETURN_NONE;
  if (cos.strides() != sin.strides()) Py_RETURN_NONE;
  int64_t n = wb.size(0);
  if (args[11] != Py_None) {
    if (!PyLong_CheckExact(args[11])) Py_RETURN_NONE;
    n = PyLong_AsLongLong(args[11]);
  }
  const int64_t layer = PyLong_AsLongLong(args[2]);
  if (PyErr_Occurred()) {
    PyErr_Clear();
    Py_RETURN_NONE;
  }
  if (n < 0 || n > wb.size(0) || n > wo.size(0) || n > rows) Py_RETURN_NONE;
  at::Tensor out;
  if (!result_like(args[10], q, &out)) Py_RETURN_NONE;
  void* const stream = PyLong_AsVoidPtr(args[12]);
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = g_rope(kc.data_ptr(), vc.data_ptr(), kc.strides().data(), q.data_ptr(), q.strides().data(), k.data_ptr(),
              k.strides().data(), v.data_ptr(), v.strides().data(), cos.data_ptr(), sin.data_ptr(), cos.strides().data(),
              out.data_ptr(), out.strides().data(), wb.data_ptr<int64_t>(), wo.data_ptr<int64_t>(), rows, n, layer,
              kc.size(1), kc.size(0), kc.size(2), q.size(1), hkv, d, code, stream);
  Py_END_ALLOW_THREADS
  return result(rc, out);
  END_HANDLE_TH_ERRORS
}

// bind(decode, decode_append, decode_bytes, prefill, prefill_bytes, rope):
// addresses of the loaded library's entry points.
PyObject* bind(PyObject*, PyObject* args) {
  PyObject* a[6];
  if (!PyArg_ParseTuple(args, "OOOOOO", &a[0], &a[1], &a[2], &a[3], &a[4], &a[5])) return nullptr;
  void* p[6];
  for (int i = 0; i < 6; ++i) {
    p[i] = PyLong_AsVoidPtr(a[i]);
    if (!p[i] && PyErr_Occurred()) return nullptr;
  }
  g_decode = reinterpret_cast<decltype(g_decode)>(p[0]);
  g_decode_append = reinterpret_cast<decltype(g_decode_append)>(p[1]);
  g_decode_bytes = reinterpret_cast<decltype(g_decode_bytes)>(p[2]);
  g_prefill = reinterpret_cast<decltype(g_prefill)>(p[3]);
  g_prefill_bytes = reinterpret_cast<decltype(g_prefill_bytes)>(p[4]);
  g_rope = reinterpret_cast<decltype(g_rope)>(p[5]);
  Py_RETURN_NONE;
}

PyMethodDef kMethods[] = {
    {"bind", bind, METH_VARARGS, nullptr},
    {"decode", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(decode)), METH_FASTCALL, nullptr},
    {"prefill", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(prefill)), METH_FASTCALL, nullptr},
    {"prefill_bytes", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(prefill_bytes)), METH_FASTCALL, nullptr},
    {"rope", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(rope)), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_host_calls", nullptr, -1, kMethods};

}  // namespace

PyMODINIT_FUNC PyInit__host_calls(void) { return PyModule_Create(&kModule); }
