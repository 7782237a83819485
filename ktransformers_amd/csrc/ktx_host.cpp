// ktx_host.cpp — the host side of the shortest calls (a CPython module, built as lib/ktx_host-<torch><interpreter>.so): checks, the result's allocation and the call into
// libktx_hip.so without an interpreter step per argument.
//
// A decode step makes these calls by the hundred, and their kernels take 4 to 12 us: in Python (ctypes converts 10 to 20 arguments, a tensor's sizes and
// strides are objects) the host took 8 to 16 us a call, and the device waited.  Every function here takes exactly the calls that it has checked — dense tensors of the
// expected types, sizes and strides on the handle's device, no dispatch or function mode — and returns None for all others: _native.py then
// goes its own way, which raises what is to be raised.  The entry points' addresses come from _native.py, so that this module needs no library of its own.
//
// Host time of a call (python, launches and, for the attention, the caller's slices), us, in Python -> here: linear of one row 8.0 -> 4.4 (its kernel 4.1 to 5.9), experts of one
// token 10.4 -> 7.0 (8.7 and more), MLA decode 16.0 -> 10.4 (7.8 and more), MLA prompt 14.8 -> 8.5 (8.2 and more).
#include <torch/csrc/autograd/python_variable.h>
#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>

#include <cstring>
#include <string>

#include "../../include/ktx_mla.h"

namespace {

typedef int (*mla_prefill_fn)(int, int, int, int, float, const void*, int64_t, int64_t, const void*, int64_t, int64_t, const void*, const void*, int64_t,
                              const void*, void*, void*, size_t, void*);
typedef size_t (*mla_prefill_bytes_fn)(int, int, int);
typedef int (*mla_decode_fn)(const ktx_mla_config*, const void*, const void*, void*, void*, int64_t, int64_t, const int32_t*, const int32_t*, const int32_t*,
                             const int32_t*, const int32_t*, int, int, const void*, const void*, void*, float*, void*, size_t, void*);
typedef int (*linear_fn)(void*, const int32_t*, int, const void*, void*, void*);
typedef int (*moe_fn)(void*, const int32_t*, int, int, const int64_t*, const float*, const void*, void*, int, void*);
typedef const char* (*error_fn)();

mla_prefill_fn g_prefill;
mla_prefill_bytes_fn g_prefill_bytes;
mla_decode_fn g_decode;
linear_fn g_linear;
moe_fn g_moe;
error_fn g_error;
PyObject* g_error_type;

// What is neither a plain strided tensor of the GPU nor its autograd wrapper (functorch's, fake, functional, conjugated, sparse, ...) is Python's.
inline const at::Tensor* plain(PyObject* o, at::ScalarType type) {
  static const c10::DispatchKeySet usual({c10::DispatchKey::CUDA, c10::DispatchKey::AutogradCUDA, c10::DispatchKey::AutocastCUDA, c10::DispatchKey::ADInplaceOrView});
  static const c10::DispatchKeySet inference({c10::DispatchKey::CUDA, c10::DispatchKey::AutocastCUDA});
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  const c10::DispatchKeySet ks = t.key_set();
  if ((ks != usual && ks != inference) || t.scalar_type() != type) return nullptr;
  return &t;
}
inline bool modes() {   // (or a transform of torch.func, inside which new tensors are wrapped)
  return c10::impl::TorchDispatchModeTLS::any_modes_set() || at::impl::torch_function_mode_enabled() ||
         c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode);
}
inline void* stream_of(const at::Tensor& t) { return (void*)c10::hip::getCurrentHIPStream(t.get_device()).stream(); }
inline PyObject* none() { Py_RETURN_NONE; }
inline bool integer(PyObject* o, int64_t& v) {
  if (!PyLong_CheckExact(o)) return false;
  v = PyLong_AsLongLong(o);
  if (v == -1 && PyErr_Occurred()) { PyErr_Clear(); return false; }
  return true;
}

struct Released {   // the interpreter, while a launch may wait for the queue, or memory for the allocator or the device
  PyThreadState* state = PyEval_SaveThread();
  ~Released() { PyEval_RestoreThread(state); }
};

// f(out, scratch, stream) into a tensor of `sizes` beside x, with `need` bytes of scratch.  None where there is no memory for them: Python's way says so, or does without.
template <class F>
PyObject* call(at::IntArrayRef sizes, const at::Tensor& x, F&& f, size_t need = 0) {
  at::Tensor out;
  int rc = 0;
  bool allocated = false;
  std::string what;
  try {
    const Released r;
    at::Tensor ws;   // (given back before the interpreter is waited for)
    out = at::empty(sizes, x.options().requires_grad(false));
    if (need) ws = at::empty({(int64_t)need}, x.options().requires_grad(false).dtype(at::kByte));
    void* stream = stream_of(x);
    allocated = true;
    rc = f(out.data_ptr(), need ? ws.data_ptr() : nullptr, stream);
  } catch (const std::exception& e) {
    if (!allocated) return none();
    what = e.what();
    rc = -1;
  }
  if (rc != 0) {
    PyErr_SetString(g_error_type, what.empty() ? g_error() : what.c_str());
    return nullptr;
  }
  return THPVariable_Wrap(std::move(out));
}

// linear(handle, K, N, device index, x): bf16 [T, K] of up to 8 rows, dense
PyObject* linear(PyObject*, PyObject* const* a, Py_ssize_t n) {
  int64_t h, K, N, dev;
  if (n != 5 || !integer(a[0], h) || !h || !integer(a[1], K) || !integer(a[2], N) || !integer(a[3], dev)) return none();
  const at::Tensor* x = plain(a[4], at::kBFloat16);
  if (!x || x->dim() != 2 || x->size(1) != K || x->size(0) < 1 || x->size(0) > 8 || x->get_device() != dev || !x->is_contiguous() || modes()) return none();
  const int T = (int)x->size(0);
  const void* xp = x->const_data_ptr();
  return call({T, N}, *x, [&](void* y, void*, void* st) { return g_linear((void*)h, nullptr, T, xp, y, st); });
}

// moe(handle, H, device index, x, ids, weights)
PyObject* moe(PyObject*, PyObject* const* a, Py_ssize_t n) {
  int64_t h, H, dev;
  if (n != 6 || !integer(a[0], h) || !h || !integer(a[1], H) || !integer(a[2], dev)) return none();
  const at::Tensor *x = plain(a[3], at::kBFloat16), *ids = plain(a[4], at::kLong), *w = plain(a[5], at::kFloat);
  if (!x || !ids || !w || ids->dim() != 2 || x->dim() != 2 || w->dim() != 2) return none();
  const int64_t T = ids->size(0), k = ids->size(1);
  if (T < 1 || T > INT32_MAX || k < 1 || k > INT32_MAX || x->size(0) != T || x->size(1) != H || w->size(0) != T || w->size(1) != k || x->get_device() != dev || ids->get_device() != dev ||
      w->get_device() != dev || !x->is_contiguous() || !ids->is_contiguous() || !w->is_contiguous() || modes())
    return none();
  const void* xp = x->const_data_ptr();
  const int64_t* ip = ids->const_data_ptr<int64_t>();
  const float* wp = w->const_data_ptr<float>();
  return call({T, H}, *x, [&](void* y, void*, void* st) { return g_moe((void*)h, nullptr, (int)T, (int)k, ip, wp, xp, y, 0, st); });
}

// mla_prefill(q_nope, q_pe, k_nope, k_pe, v_t, kv_len, sm_scale)
PyObject* mla_prefill(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 7) return none();
  const at::Tensor* t[5];
  for (int i = 0; i < 5; i++) {
    t[i] = plain(a[i], at::kBFloat16);
    if (!t[i] || t[i]->dim() != (i == 3 ? 2 : 3) || t[i]->stride(-1) != 1) return none();
  }
  int64_t kv;
  if (!integer(a[5], kv) || kv < INT32_MIN || kv > INT32_MAX || !PyFloat_CheckExact(a[6]) || modes()) return none();
  const at::Tensor &qn = *t[0], &qp = *t[1], &kn = *t[2], &kp = *t[3], &v = *t[4];
  const int64_t T = qn.size(0), H = qn.size(1), pad = kn.size(1);
  if (T < 1 || H < 1 || T > INT32_MAX || H > INT32_MAX || pad > INT32_MAX || qn.size(2) != 128 || qp.size(2) != 64 || kn.size(0) != H || kn.size(2) != 128 || v.size(0) != H || v.size(1) != 128 ||
      v.size(2) != pad || kp.size(1) != 64 || !kn.is_contiguous() || !v.is_contiguous())
    return none();
  const float scale = (float)PyFloat_AS_DOUBLE(a[6]);
  const size_t need = g_prefill_bytes((int)T, (int)H, (int)kv);
  return call({T, H, 128}, qn, [&](void* y, void* ws, void* st) {
    return g_prefill((int)T, (int)H, (int)kv, (int)pad, scale, qn.const_data_ptr(), qn.stride(0), qn.stride(1), qp.const_data_ptr(), qp.stride(0), qp.stride(1),
                     kn.const_data_ptr(), kp.const_data_ptr(), kp.stride(0), v.const_data_ptr(), y, ws, need, st);
  }, need);
}

// mla_decode(config, most query tokens, q_nope, q_pe, ckv, k_pe, qo_indptr, kv_indptr, kv_indices | None, kv_len, bsz | None, workspace)
PyObject* mla_decode(PyObject*, PyObject* const* a, Py_ssize_t n) {
  int64_t most;
  ktx_mla_config c;
  if (n != 12 || !integer(a[1], most)) return none();
  {   // a copy: another thread's plan may replace the wrapper's while the interpreter is released
    Py_buffer b;
    if (PyObject_GetBuffer(a[0], &b, PyBUF_SIMPLE) != 0) { PyErr_Clear(); return none(); }
    const bool whole = b.len == (Py_ssize_t)sizeof c;
    if (whole) std::memcpy(&c, b.buf, sizeof c);
    PyBuffer_Release(&b);
    if (!whole) return none();
  }
  const int64_t page = c.page_size;
  const at::Tensor *qn = plain(a[2], at::kBFloat16), *qp = plain(a[3], at::kBFloat16), *ckv = plain(a[4], at::kBFloat16), *kpe = plain(a[5], at::kBFloat16);
  const at::Tensor* ix[5];
  for (int i = 0; i < 5; i++) {
    ix[i] = a[6 + i] == Py_None && (i == 2 || i == 4) ? nullptr : plain(a[6 + i], at::kInt);
    if (!ix[i] && a[6 + i] != Py_None) return none();
  }
  const at::Tensor* ws = plain(a[11], at::kByte);
  if (!qn || !qp || !ckv || !kpe || !ix[0] || !ix[1] || !ix[3] || !ws || qn->dim() != 3 || ckv->dim() < 2 || kpe->dim() < 2 || modes()) return none();
  const int64_t T = qn->size(0), H = qn->size(1), dc = qn->size(2), cs = ckv->stride(-2), ps = kpe->stride(-2), batch = ix[0]->numel() - 1;
  if (T < 1 || T > most || T > INT32_MAX || batch > INT32_MAX || !qn->is_contiguous() || !qp->is_contiguous() || ckv->stride(-1) != 1 || kpe->stride(-1) != 1 || ckv->stride(0) != cs * page ||
      kpe->stride(0) != ps * page)
    return none();
  return call({T, H, dc}, *qn, [&](void* y, void*, void* st) {
    return g_decode(&c, qn->const_data_ptr(), qp->const_data_ptr(), (void*)ckv->const_data_ptr(), (void*)kpe->const_data_ptr(), cs, ps, ix[0]->const_data_ptr<int32_t>(),
                    ix[1]->const_data_ptr<int32_t>(), ix[2] ? ix[2]->const_data_ptr<int32_t>() : nullptr, ix[3]->const_data_ptr<int32_t>(),
                    ix[4] ? ix[4]->const_data_ptr<int32_t>() : nullptr, (int)batch, (int)T, nullptr, nullptr, y, nullptr, (void*)ws->const_data_ptr(), (size_t)ws->numel(), st);
  });
}

// bind(error type, last_error, linear, moe, mla_prefill_ws, mla_decode, mla_prefill_workspace_bytes): the entry points' addresses
PyObject* bind(PyObject*, PyObject* const* a, Py_ssize_t n) {
  int64_t p[6];
  if (n != 7) { PyErr_SetString(PyExc_TypeError, "bind: 7 arguments"); return nullptr; }
  for (int i = 0; i < 6; i++)
    if (!integer(a[i + 1], p[i])) { PyErr_SetString(PyExc_TypeError, "bind: addresses"); return nullptr; }
  Py_INCREF(a[0]);
  Py_XDECREF(g_error_type);
  g_error_type = a[0];
  g_error = (error_fn)p[0]; g_linear = (linear_fn)p[1]; g_moe = (moe_fn)p[2]; g_prefill = (mla_prefill_fn)p[3]; g_decode = (mla_decode_fn)p[4]; g_prefill_bytes = (mla_prefill_bytes_fn)p[5];
  Py_RETURN_NONE;
}

PyMethodDef methods[] = {{"bind", (PyCFunction)(void (*)(void))bind, METH_FASTCALL, nullptr},
                         {"linear", (PyCFunction)(void (*)(void))linear, METH_FASTCALL, nullptr},
                         {"moe", (PyCFunction)(void (*)(void))moe, METH_FASTCALL, nullptr},
                         {"mla_prefill", (PyCFunction)(void (*)(void))mla_prefill, METH_FASTCALL, nullptr},
                         {"mla_decode", (PyCFunction)(void (*)(void))mla_decode, METH_FASTCALL, nullptr},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "ktx_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_ktx_host(void) { return PyModule_Create(&module); }
