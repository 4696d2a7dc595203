// The operators' host side, native: one call from Python checks the tensors of a plain call, allocates what it returns and the scratch, and
// goes through the C ABI.  Anything that is not a plain call -- another layout, a mistake, a tensor subclass -- returns None, and the Python
// binding that called does it (and raises what it always raised).  No kernel and no rule lives here.
//
// What bounds the smallest calls is the host: torch.empty takes 2 us, a ctypes call of 25 arguments 4, beside 3 for a launch.  A forward without
// gradients 15.4 -> 10.0 us of the host's time; forward and backward, on a machine where the autograd engine's hand-over to its thread is slow:
// B4 H8 N512 D64 117 -> 110 us, Co-RoPE B2 Hq8 Hkv2 N512 D64 134 -> 105, B2 Hq16 Hkv8 N82 D128 127 -> 104.
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/pycfunction_helpers.h>
#include <ATen/ATen.h>
#include <torch/version.h>

#include "../../include/corope_amd.h"

namespace {

// Entry points of the library in use, by address (the order of host_calls in _lib.py).
struct Table {
  decltype(&corope_rope_attn_fwd_keep) fwd_keep;
  decltype(&corope_rope_attn_bwd_rotated) bwd;
  decltype(&corope_gqa_fwd) gqa_fwd, gqa_fwd_f16;
  decltype(&corope_gqa_bwd) gqa_bwd, gqa_bwd_f16;
};
constexpr int kEntries = sizeof(Table) / sizeof(void*);

struct NoGil {
  PyThreadState* state = PyEval_SaveThread();
  ~NoGil() { PyEval_RestoreThread(state); }
};

// A tensor the kernels can be handed as it is: a plain strided GPU tensor on `device` (the current one) that no transform has wrapped.
const at::Tensor* plain(PyObject* o, int device) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  if (!t.defined() || !t.is_cuda() || t.get_device() != device || t.layout() != at::kStrided || !t.has_storage()) return nullptr;
  const auto ks = t.key_set();
  if (ks.has(c10::DispatchKey::FuncTorchBatched) || ks.has(c10::DispatchKey::FuncTorchGradWrapper) || ks.has(c10::DispatchKey::Batched) ||
      ks.has(c10::DispatchKey::Functionalize) || ks.has(c10::DispatchKey::Python) || t.is_neg() || t.is_conj())
    return nullptr;
  return &t;
}

bool aligned16(const at::Tensor& t) { return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0; }

// (batch, head, row) strides of a contiguous tensor, or of a view that the kernels read where it lies.
bool strides_of(const at::Tensor& t, int64_t (&st)[3]) {
  if (!aligned16(t)) return false;
  const int64_t D = t.size(3), N = t.size(2);
  if (t.is_contiguous()) {   // (an axis of length 1 may say otherwise)
    st[0] = t.size(1) * N * D, st[1] = N * D, st[2] = D;
    return true;
  }
  st[0] = t.stride(0), st[1] = t.stride(1), st[2] = t.stride(2);
  return t.stride(3) == 1 && st[2] >= D && st[0] >= 0 && st[1] >= 0 && st[0] % 8 == 0 && st[1] % 8 == 0 && st[2] % 8 == 0 && N * st[2] * 2 < (1ll << 32);
}

bool same_kind(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v) {
  if (q.dim() != 4 || k.dim() != 4 || v.dim() != 4 || q.numel() == 0 || k.numel() == 0) return false;
  const auto type = q.scalar_type();
  return (type == at::kBFloat16 || type == at::kHalf) && k.scalar_type() == type && v.scalar_type() == type && k.sizes() == v.sizes() &&
         q.size(0) == k.size(0) && q.size(2) == k.size(2) && q.size(3) == k.size(3) && q.size(1) % k.size(1) == 0 && q.size(0) < (1 << 30) &&
         q.size(1) < (1 << 30) && q.size(2) < (1 << 30);
}

bool table_ok(const at::Tensor& f, int64_t N, int64_t D) {
  return f.dim() == 2 && f.scalar_type() == at::kFloat && f.size(0) >= N && f.size(1) >= D / 2 && f.stride(1) == 1 && f.stride(0) % 4 == 0 && aligned16(f);
}

// Scratch for cut blocks, from the caller: a byte tensor, or None (undefined: nothing is cut).
bool parts_of(PyObject* o, int device, at::Tensor& parts) {
  if (o == Py_None) return true;
  const at::Tensor* t = plain(o, device);
  if (t == nullptr || !t->is_contiguous()) return false;
  parts = *t;
  return true;
}

void* data(const at::Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }
float* floats(const at::Tensor& t) { return static_cast<float*>(data(t)); }

PyObject* pack(std::initializer_list<at::Tensor> ts) {
  PyObject* out = PyTuple_New((Py_ssize_t)ts.size());
  if (out == nullptr) return nullptr;
  Py_ssize_t i = 0;
  for (const auto& t : ts) {
    PyObject* o = t.defined() ? THPVariable_Wrap(t) : (Py_INCREF(Py_None), Py_None);
    if (o == nullptr) {
      Py_DECREF(out);
      return nullptr;
    }
    PyTuple_SET_ITEM(out, i++, o);
  }
  return out;
}

const Table* table_of(PyObject* capsule) { return static_cast<const Table*>(PyCapsule_GetPointer(capsule, "corope_table")); }

#define COROPE_ARGS(n)                                                                  \
  if (nargs != (n)) {                                                                   \
    PyErr_Format(PyExc_TypeError, "%s takes %d arguments (got %zd)", __func__, n, nargs); \
    return nullptr;                                                                     \
  }

// make_table(addresses): the capsule that the other functions take
PyObject* make_table(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  COROPE_ARGS(kEntries)
  auto* t = new Table;
  for (int i = 0; i < kEntries; ++i) reinterpret_cast<void**>(t)[i] = PyLong_AsVoidPtr(args[i]);
  if (PyErr_Occurred()) {
    delete t;
    return nullptr;
  }
  return PyCapsule_New(t, "corope_table", nullptr);   // (lives as long as the library: until the process ends)
}

// rope_forward(table, q, k, v, cos, sin, causal, sm_scale, rotated, exact, keep, device, stream, parts)
//   -> None | status | (o, lse, q_rot or None, k_rot or None, v: a contiguous one where keep asks for it)
PyObject* rope_forward(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  COROPE_ARGS(14)
  const Table* tab = table_of(args[0]);
  const int causal = PyObject_IsTrue(args[6]), rotated = PyObject_IsTrue(args[8]), exact = PyObject_IsTrue(args[9]), keep = PyObject_IsTrue(args[10]);
  const double sm_scale = PyFloat_AsDouble(args[7]);
  const int device = (int)PyLong_AsLong(args[11]);
  void* stream = PyLong_AsVoidPtr(args[12]);
  if (tab == nullptr || PyErr_Occurred()) return nullptr;
  const at::Tensor* x[5];
  for (int i = 0; i < 5; ++i)
    if ((x[i] = plain(args[1 + i], device)) == nullptr) Py_RETURN_NONE;
  const at::Tensor &q = *x[0], &k = *x[1], &v = *x[2], &fc = *x[3], &fs = *x[4];
  if (!same_kind(q, k, v)) Py_RETURN_NONE;
  const int B = (int)q.size(0), H = (int)q.size(1), Hkv = (int)k.size(1), N = (int)q.size(2), D = (int)q.size(3);
  int64_t qs[3], ks[3], vs[3];
  if ((D != 64 && D != 128 && D != 256) || !table_ok(fc, N, D) || !table_ok(fs, N, D) || fc.stride(0) != fs.stride(0) || !strides_of(q, qs) ||
      !strides_of(k, ks) || !strides_of(v, vs))
    Py_RETURN_NONE;
  if (keep && !rotated && !v.is_contiguous()) Py_RETURN_NONE;
  const auto opts = q.options().requires_grad(false), fopts = opts.dtype(at::kFloat);
  at::Tensor o, lse, v_keep, q_rot, k_rot, kmax, parts;
  if (!parts_of(args[13], device, parts)) Py_RETURN_NONE;
  o = at::empty({B, H, N, D}, opts);
  lse = at::empty({B, H, N}, fopts);
  if (rotated) {
    k_rot = at::empty({B, Hkv, N, D}, opts);
    if (keep) q_rot = at::empty({B, H, N, D}, opts);
    if (keep && !v.is_contiguous()) v_keep = at::empty({B, Hkv, N, D}, opts);
    if (!exact) kmax = at::empty({B, Hkv, (N + 63) / 64}, fopts);
  }
  int rc;
  {
    NoGil free;
    rc = tab->fwd_keep(q.data_ptr(), qs, k.data_ptr(), ks, v.data_ptr(), vs, floats(fc), floats(fs), fc.stride(0), o.data_ptr(), floats(lse), data(q_rot),
                      data(k_rot), floats(kmax), B, H, Hkv, N, D, (float)sm_scale, causal, q.scalar_type() == at::kHalf, data(parts), parts.defined() ? (int64_t)parts.nbytes() : 0, data(v_keep), stream);
  }
  if (rc != 0) return PyLong_FromLong(rc);
  return pack({o, lse, q_rot, keep ? k_rot : at::Tensor(), v_keep.defined() ? v_keep : v});
  END_HANDLE_TH_ERRORS
}

// rope_backward(table, q_rot, k_rot, v, o, d_o, lse, cos, sin, causal, sm_scale, device, stream, parts) -> None | status | (dq, dk, dv)
PyObject* rope_backward(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  COROPE_ARGS(14)
  const Table* tab = table_of(args[0]);
  const int causal = PyObject_IsTrue(args[9]);
  const double sm_scale = PyFloat_AsDouble(args[10]);
  const int device = (int)PyLong_AsLong(args[11]);
  void* stream = PyLong_AsVoidPtr(args[12]);
  if (tab == nullptr || PyErr_Occurred()) return nullptr;
  const at::Tensor* x[8];
  for (int i = 0; i < 8; ++i)
    if ((x[i] = plain(args[1 + i], device)) == nullptr) Py_RETURN_NONE;
  const at::Tensor &q = *x[0], &k = *x[1], &v = *x[2], &o = *x[3], &lse = *x[5], &fc = *x[6], &fs = *x[7];
  if (!same_kind(q, k, v) || o.sizes() != q.sizes() || x[4]->sizes() != q.sizes() || x[4]->scalar_type() != q.scalar_type()) Py_RETURN_NONE;
  for (const at::Tensor* t : {x[0], x[1], x[2], x[3], x[5]})   // (what saved-tensor hooks handed back may lie otherwise)
    if (!t->is_contiguous() || !aligned16(*t)) Py_RETURN_NONE;
  const int B = (int)q.size(0), H = (int)q.size(1), Hkv = (int)k.size(1), N = (int)q.size(2), D = (int)q.size(3);
  if (o.scalar_type() != q.scalar_type() || lse.scalar_type() != at::kFloat || lse.numel() != (int64_t)B * H * N || !table_ok(fc, N, D) || !table_ok(fs, N, D) ||
      fc.stride(0) != fs.stride(0))
    Py_RETURN_NONE;
  at::Tensor d_o = *x[4];
  int64_t ds[3];
  bool view = !d_o.is_contiguous();
  if (view && (D > 128 || !strides_of(d_o, ds))) {   // what the kernels cannot read where it lies is copied
    d_o = d_o.contiguous();
    view = false;
  }
  if (!aligned16(d_o)) Py_RETURN_NONE;
  at::Tensor parts;
  if (!parts_of(args[13], device, parts)) Py_RETURN_NONE;
  const auto opts = q.options().requires_grad(false);
  at::Tensor dq = at::empty({B, H, N, D}, opts), dk = at::empty({B, Hkv, N, D}, opts), dv = at::empty({B, Hkv, N, D}, opts);
  at::Tensor delta = at::empty({B, H, N}, opts.dtype(at::kFloat));
  int rc;
  {
    NoGil free;
    rc = tab->bwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), nullptr, o.data_ptr(), d_o.data_ptr(), view ? ds : nullptr, floats(lse), floats(delta), floats(fc),
                  floats(fs), fc.stride(0), dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), B, H, Hkv, N, D, (float)sm_scale, causal,
                  q.scalar_type() == at::kHalf, data(parts), parts.defined() ? (int64_t)parts.nbytes() : 0, stream);
  }
  if (rc != 0) return PyLong_FromLong(rc);
  return pack({dq, dk, dv});
  END_HANDLE_TH_ERRORS
}

// gqa_forward(table, q, k, v, sm_scale, theta, device, stream) -> None | status | (o,)
PyObject* gqa_forward(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  COROPE_ARGS(8)
  const Table* tab = table_of(args[0]);
  const double sm_scale = PyFloat_AsDouble(args[4]), theta = PyFloat_AsDouble(args[5]);
  const int device = (int)PyLong_AsLong(args[6]);
  void* stream = PyLong_AsVoidPtr(args[7]);
  if (tab == nullptr || PyErr_Occurred()) return nullptr;
  const at::Tensor* x[3];
  for (int i = 0; i < 3; ++i)
    if ((x[i] = plain(args[1 + i], device)) == nullptr || !x[i]->is_contiguous() || !aligned16(*x[i])) Py_RETURN_NONE;
  const at::Tensor &q = *x[0], &k = *x[1], &v = *x[2];
  if (!same_kind(q, k, v)) Py_RETURN_NONE;
  const int B = (int)q.size(0), H = (int)q.size(1), Hkv = (int)k.size(1), N = (int)q.size(2), D = (int)q.size(3);
  at::Tensor o = at::empty({B, H, N, D}, q.options().requires_grad(false));
  int rc;
  {
    NoGil free;
    rc = (q.scalar_type() == at::kHalf ? tab->gqa_fwd_f16 : tab->gqa_fwd)(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), B, H, Hkv, N, D,
                                                                         (float)sm_scale, (float)theta, stream);
  }
  if (rc != 0) return PyLong_FromLong(rc);
  return pack({o});
  END_HANDLE_TH_ERRORS
}

// gqa_backward(table, q, k, v, o, d_o, workspace, sm_scale, theta, device, stream) -> None | status | (dq, dk, dv)
PyObject* gqa_backward(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  COROPE_ARGS(11)
  const Table* tab = table_of(args[0]);
  const double sm_scale = PyFloat_AsDouble(args[7]), theta = PyFloat_AsDouble(args[8]);
  const int device = (int)PyLong_AsLong(args[9]);
  void* stream = PyLong_AsVoidPtr(args[10]);
  if (tab == nullptr || PyErr_Occurred()) return nullptr;
  const at::Tensor* x[6];
  for (int i = 0; i < 6; ++i)
    if ((x[i] = plain(args[1 + i], device)) == nullptr || !x[i]->is_contiguous() || !aligned16(*x[i])) Py_RETURN_NONE;
  const at::Tensor &q = *x[0], &k = *x[1], &v = *x[2], &o = *x[3], &d_o = *x[4], &ws = *x[5];
  if (!same_kind(q, k, v) || o.sizes() != q.sizes() || d_o.sizes() != q.sizes() || o.scalar_type() != q.scalar_type() || d_o.scalar_type() != q.scalar_type())
    Py_RETURN_NONE;
  const int B = (int)q.size(0), H = (int)q.size(1), Hkv = (int)k.size(1), N = (int)q.size(2), D = (int)q.size(3);
  const auto opts = q.options().requires_grad(false);
  at::Tensor dq = at::empty({B, H, N, D}, opts), dk = at::empty({B, Hkv, N, D}, opts), dv = at::empty({B, Hkv, N, D}, opts);
  int rc;
  {
    NoGil free;
    rc = (q.scalar_type() == at::kHalf ? tab->gqa_bwd_f16 : tab->gqa_bwd)(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), d_o.data_ptr(), dq.data_ptr(),
                                                                         dk.data_ptr(), dv.data_ptr(), B, H, Hkv, N, D, (float)sm_scale, (float)theta,
                                                                         ws.data_ptr(), (int64_t)ws.nbytes(), stream);
  }
  if (rc != 0) return PyLong_FromLong(rc);
  return pack({dq, dk, dv});
  END_HANDLE_TH_ERRORS
}

#define COROPE_METHOD(f) {#f, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(f)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {COROPE_METHOD(make_table), COROPE_METHOD(rope_forward), COROPE_METHOD(rope_backward), COROPE_METHOD(gqa_forward),
                         COROPE_METHOD(gqa_backward), {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "corope_host_calls", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

extern "C" __attribute__((visibility("default"))) PyObject* PyInit_corope_host_calls(void) {
  PyObject* m = PyModule_Create(&module);
  // (the tensors' layout is that of the torch this was built against: the loader compares)
  if (m != nullptr && PyModule_AddStringConstant(m, "torch_version", TORCH_VERSION) != 0) Py_CLEAR(m);
  return m;
}
