// The per-forward host work of the Python modules in native code: a CPython extension
// over libtorch that allocates a call's outputs and workspace and enters libtmoe's C ABI
// (whose addresses bind() receives from the ctypes binding, so that both use one
// library), with X's device current. Checks of shapes, dtypes and devices stay with the
// Python callers.
//
// Why: at decode sizes a forward's kernels take 8.5-11 us, and the same steps through
// ctypes and torch's Python API took 21 us a layer (the packed-weights key 6.0, the two
// allocations 2.2, the ctypes call 3.4 of which 2.7 are the launch, stream and device 3.1).
// Here a layer takes 7.5-8.5 us of host time, launch included, so that one-launch forwards
// follow each other at the kernel's pace: decode at T = 1 and 32 22.8 -> 12 us.
#include <ATen/ops/empty.h>
#include <c10/core/DeviceGuard.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstdint>
#include <vector>

#include "tmoe.h"

namespace {

struct Entry {
  decltype(&tmoe_workspace_bytes) workspace_bytes;
  decltype(&tmoe_signal_status) signal_status;
  decltype(&tmoe_forward_epi) forward_epi;
  decltype(&tmoe_forward_glu) forward_glu;
  decltype(&tmoe_rmsnorm_rows) rmsnorm_rows;
} g_lib{};
PyObject *g_gen, *g_alias;   // "_tmoe_gen", "_tmoe_alias" (module.TrackedParameter)

bool bad_args(Py_ssize_t n, Py_ssize_t want, const char* who) {
  if (n == want) return false;
  PyErr_Format(PyExc_TypeError, "%s: %zd arguments, %zd expected", who, n, want);
  return true;
}
const at::Tensor& tensor(PyObject* o) {
  if (!THPVariable_Check(o)) throw torch::TypeError("a tensor expected");
  return THPVariable_Unpack(o);
}
void* opt_ptr(PyObject* o) { return o == Py_None ? nullptr : tensor(o).data_ptr(); }
void* address(PyObject* o) {
  void* p = PyLong_AsVoidPtr(o);
  if (PyErr_Occurred()) throw python_error();
  return p;
}
int64_t integer(PyObject* o) {
  const int64_t v = PyLong_AsLongLong(o);
  if (v == -1 && PyErr_Occurred()) throw python_error();
  return v;
}
at::Tensor bytes_like(const at::Tensor& t, size_t n) {
  return at::empty({static_cast<int64_t>(n ? n : 1)}, t.options().dtype(at::kByte));
}
PyObject* none() {
  Py_INCREF(Py_None);
  return Py_None;
}

PyObject* bind(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (bad_args(n, 5, "bind")) return nullptr;
  g_lib.workspace_bytes = reinterpret_cast<decltype(g_lib.workspace_bytes)>(address(a[0]));
  g_lib.signal_status = reinterpret_cast<decltype(g_lib.signal_status)>(address(a[1]));
  g_lib.forward_epi = reinterpret_cast<decltype(g_lib.forward_epi)>(address(a[2]));
  g_lib.forward_glu = reinterpret_cast<decltype(g_lib.forward_glu)>(address(a[3]));
  g_lib.rmsnorm_rows = reinterpret_cast<decltype(g_lib.rmsnorm_rows)>(address(a[4]));
  return none();
  END_HANDLE_TH_ERRORS
}

// param_key(tensors): bytes that differ when a tensor's storage address, version counter,
// dtype or device changed, or (TrackedParameter) its `.data` was assigned or written
// through.
PyObject* param_key(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (bad_args(n, 1, "param_key")) return nullptr;
  if (!PyTuple_Check(a[0])) throw torch::TypeError("param_key: a tuple expected");
  struct Rec {
    uint64_t ptr, version;
    int64_t gen;
    uint64_t alias_version;
    int32_t dtype, device;
  };
  const Py_ssize_t m = PyTuple_GET_SIZE(a[0]);
  std::vector<Rec> recs(m);
  for (Py_ssize_t i = 0; i < m; ++i) {
    PyObject* o = PyTuple_GET_ITEM(a[0], i);
    const at::Tensor& t = tensor(o);
    Rec& r = recs[i];
    r.ptr = reinterpret_cast<uint64_t>(t.data_ptr());
    r.version = t._version();
    r.gen = 0;
    r.alias_version = 0;
    r.dtype = static_cast<int32_t>(t.scalar_type());
    r.device = static_cast<int32_t>(t.device().type()) << 16 | (t.device().index() & 0xffff);
    PyObject* d = PyObject_GenericGetDict(o, nullptr);
    if (!d) {
      PyErr_Clear();
      continue;
    }
    if (PyObject* g = PyDict_GetItemWithError(d, g_gen)) r.gen = PyLong_AsLongLong(g);
    PyObject* al = PyDict_GetItemWithError(d, g_alias);
    if (al && THPVariable_Check(al)) r.alias_version = THPVariable_Unpack(al)._version();
    Py_DECREF(d);
    if (PyErr_Occurred()) return nullptr;
  }
  return PyBytes_FromStringAndSize(reinterpret_cast<const char*>(recs.data()),
                                   static_cast<Py_ssize_t>(m * sizeof(Rec)));
  END_HANDLE_TH_ERRORS
}

// signal(plan): tmoe_signal_status with clearing; its return code.
PyObject* signal_(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (bad_args(n, 1, "signal")) return nullptr;
  uint32_t mask = 0;
  return PyLong_FromLong(
      g_lib.signal_status(static_cast<const tmoe_plan*>(address(a[0])), 1, &mask));
  END_HANDLE_TH_ERRORS
}

// forward(plan, X, packed, out or None, d_out, k, E, epi, epi_a, epi_b, stream):
// tmoe_forward_epi on the contiguous (T, d_in) X with a workspace of its own. k > 0
// returns the routing, E > 0 the logits. (out, idx, w, logits), or a negative return code.
PyObject* forward(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (bad_args(n, 11, "forward")) return nullptr;
  const auto* plan = static_cast<const tmoe_plan*>(address(a[0]));
  const at::Tensor& x = tensor(a[1]);
  const at::Tensor& packed = tensor(a[2]);
  const c10::DeviceGuard guard(x.device());
  const int64_t T = x.size(0), d_out = integer(a[4]), k = integer(a[5]), E = integer(a[6]);
  const int epi = static_cast<int>(integer(a[7]));
  void *ea = opt_ptr(a[8]), *eb = opt_ptr(a[9]), *stream = address(a[10]);
  at::Tensor out = a[3] == Py_None ? at::empty({T, d_out}, x.options()) : tensor(a[3]);
  at::Tensor idx, w, lg;
  if (k > 0) {
    idx = at::empty({T, k}, x.options().dtype(at::kInt));
    w = at::empty({T, k}, x.options().dtype(at::kFloat));
  }
  if (E > 0) lg = at::empty({T, E}, x.options().dtype(at::kFloat));
  const size_t nws = g_lib.workspace_bytes(plan, T);
  at::Tensor ws = bytes_like(x, nws);
  void *xp = x.data_ptr(), *pp = packed.data_ptr(), *op = out.data_ptr(), *wp = ws.data_ptr();
  auto* ip = k > 0 ? static_cast<int32_t*>(idx.data_ptr()) : nullptr;
  auto* wtp = k > 0 ? static_cast<float*>(w.data_ptr()) : nullptr;
  auto* lp = E > 0 ? static_cast<float*>(lg.data_ptr()) : nullptr;
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = g_lib.forward_epi(plan, xp, T, pp, op, ip, wtp, lp, wp, nws, epi, ea, eb, stream);
  Py_END_ALLOW_THREADS
  if (rc < 0) return PyLong_FromLong(rc);
  PyObject* r = PyTuple_New(4);
  if (!r) return nullptr;
  PyObject* o = a[3];
  if (o == Py_None) o = THPVariable_Wrap(std::move(out));
  else Py_INCREF(o);
  PyTuple_SET_ITEM(r, 0, o);
  PyTuple_SET_ITEM(r, 1, k > 0 ? THPVariable_Wrap(std::move(idx)) : none());
  PyTuple_SET_ITEM(r, 2, k > 0 ? THPVariable_Wrap(std::move(w)) : none());
  PyTuple_SET_ITEM(r, 3, E > 0 ? THPVariable_Wrap(std::move(lg)) : none());
  return r;
  END_HANDLE_TH_ERRORS
}

// glu(plan, X, packed_gate, packed_up, d_out, stream): tmoe_forward_glu with workspaces
// of its own; out (T, d_out), or a negative return code.
PyObject* glu(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (bad_args(n, 6, "glu")) return nullptr;
  const auto* plan = static_cast<const tmoe_plan*>(address(a[0]));
  const at::Tensor& x = tensor(a[1]);
  const c10::DeviceGuard guard(x.device());
  void *pg = tensor(a[2]).data_ptr(), *pu = tensor(a[3]).data_ptr();
  const int64_t T = x.size(0);
  void* stream = address(a[5]);
  at::Tensor out = at::empty({T, integer(a[4])}, x.options());
  const size_t nws = g_lib.workspace_bytes(plan, T);
  at::Tensor wg = bytes_like(x, nws), wu = bytes_like(x, nws);
  void *xp = x.data_ptr(), *op = out.data_ptr(), *wgp = wg.data_ptr(), *wup = wu.data_ptr();
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = g_lib.forward_glu(plan, xp, T, pg, pu, op, wgp, wup, nws, stream);
  Py_END_ALLOW_THREADS
  if (rc < 0) return PyLong_FromLong(rc);
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// rmsnorm(X, weight, eps, dtype code, out or None, stream): tmoe_rmsnorm_rows on the
// contiguous (T, d) X; out, or a negative return code.
PyObject* rmsnorm(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (bad_args(n, 6, "rmsnorm")) return nullptr;
  const at::Tensor& x = tensor(a[0]);
  const c10::DeviceGuard guard(x.device());
  void* wp = tensor(a[1]).data_ptr();
  const double eps = PyFloat_AsDouble(a[2]);
  if (eps == -1.0 && PyErr_Occurred()) return nullptr;
  const int dt = static_cast<int>(integer(a[3]));
  void* stream = address(a[5]);
  at::Tensor y = a[4] == Py_None ? at::empty(x.sizes(), x.options()) : tensor(a[4]);
  void *xp = x.data_ptr(), *yp = y.data_ptr();
  const int64_t T = x.size(0), d = x.size(1);
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = g_lib.rmsnorm_rows(xp, T, d, wp, static_cast<float>(eps), dt, yp, stream);
  Py_END_ALLOW_THREADS
  if (rc < 0) return PyLong_FromLong(rc);
  if (a[4] != Py_None) {
    Py_INCREF(a[4]);
    return a[4];
  }
  return THPVariable_Wrap(std::move(y));
  END_HANDLE_TH_ERRORS
}

PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_tmoe_native", nullptr, -1, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__tmoe_native() {
  static PyMethodDef methods[] = {
      {"bind", (PyCFunction)(void (*)())bind, METH_FASTCALL, nullptr},
      {"param_key", (PyCFunction)(void (*)())param_key, METH_FASTCALL, nullptr},
      {"signal", (PyCFunction)(void (*)())signal_, METH_FASTCALL, nullptr},
      {"forward", (PyCFunction)(void (*)())forward, METH_FASTCALL, nullptr},
      {"glu", (PyCFunction)(void (*)())glu, METH_FASTCALL, nullptr},
      {"rmsnorm", (PyCFunction)(void (*)())rmsnorm, METH_FASTCALL, nullptr},
      {nullptr, nullptr, 0, nullptr}};
  g_gen = PyUnicode_InternFromString("_tmoe_gen");
  g_alias = PyUnicode_InternFromString("_tmoe_alias");
  if (!g_gen || !g_alias) return nullptr;
  g_module.m_methods = methods;
  PyObject* m = PyModule_Create(&g_module);
  if (m && PyModule_AddStringConstant(m, "built_for", TMOE_NATIVE_TAG) < 0) {
    Py_DECREF(m);
    return nullptr;
  }
  return m;
}
