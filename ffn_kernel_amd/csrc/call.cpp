// Python's way into the C ABI for the usual call: exact torch tensors on the current GPU, nn.Linear.weight.T views, rows the
// fast kernels address as they are.  Checks, allocations and the foreign call in one C function; anything else - another layout
// or device, a wrong argument - comes back as NotImplemented, and ops.py, which holds the rules and the error messages, takes it.
// What it is for: calls whose kernels are short are bound by the host, and the same steps in Python (three to eight tensors
// checked one attribute at a time, two to nine torch.empty calls, ctypes) were more than the launches.  Host time per call, us,
// in Python -> here, K = N = 256: MaskedLinear forward 16.2 -> 10.0 at M = 100, 18.1 -> 11.9 at M = 1 (of which 3.3 are
// Function.apply), forward + backward 145 -> 83 (of which 76 are autograd's: its worker thread ran the Python of the backward
// at a third of the speed); MaskedFFN forward 29.5 -> 16.0, forward + backward 259 -> 182.
#include <Python.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/object_ptr.h>
#include <ATen/ops/empty.h>
#include <ATen/ops/empty_strided.h>

#include "../../include/ffnk.h"

namespace {

struct Library {
  decltype(&ffnk_workspace_bytes) workspace_bytes;
  decltype(&ffnk_masked_ffn_can_save) can_save;
  decltype(&ffnk_route) route;
  decltype(&ffnk_masked_linear_fwd_routed) linear_fwd, linear_fwd_routing;
  decltype(&ffnk_masked_linear_bwd_routed) linear_bwd;
  decltype(&ffnk_masked_ffn_fwd_routed) ffn_fwd, ffn_fwd_routing;
  decltype(&ffnk_masked_ffn_bwd_routed) ffn_bwd;
} lib;
PyObject* routing_address = nullptr;    // (routing or None, mask, M, stream) -> address of a Partition, or 0
PyObject* ffn_bwd_workspace = nullptr;  // (a, d, h, row stride of the upstream gradient) -> workspace tensor
PyObject* check = nullptr;              // (return code, function name): raises
int64_t routed_min_rows = 0;            // below: no partition is shared

// _lib.PartitionStruct: memory for a row partition, and whether a launch that fills it has been made.
struct Partition {
  ffnk_routing_t routing;
  int32_t made;
};
const ffnk_routing_t* routing_of(const Partition* p) { return p ? &p->routing : nullptr; }

const uint16_t* in(const at::Tensor& t) { return static_cast<const uint16_t*>(t.const_data_ptr()); }
uint16_t* out(const at::Tensor& t) { return static_cast<uint16_t*>(t.mutable_data_ptr()); }

struct WithoutGil {
  PyThreadState* state = PyEval_SaveThread();
  ~WithoutGil() { PyEval_RestoreThread(state); }
};

// The foreign call without the GIL, as ctypes makes it.  f reads the tensors' addresses, and torch throws where one has none (an
// output that a dispatch mode made a fake tensor): the error is made a Python one by the caller, which needs the GIL back.
template <class F>
bool run(const char* name, F&& f) {
  int rc;
  {
    WithoutGil released;
    rc = f();
  }
  if (rc == 0) return true;
  PyObject* r = PyObject_CallFunction(check, "is", rc, name);
  Py_XDECREF(r);
  if (r) PyErr_SetString(PyExc_RuntimeError, name);
  return false;
}

// The tensors of a call; `ok` goes false at the first one that is not plain.
struct Call {
  bool ok = true;
  int device = -1;
  int64_t M = 0;
  void* stream = nullptr;

  const at::Tensor* strided(PyObject* o, at::ScalarType type, int64_t dims) {
    if (!ok || !THPVariable_CheckExact(o)) return fail();
    const at::Tensor& t = THPVariable_Unpack(o);
    if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || t.scalar_type() != type || t.dim() != dims || !t.has_storage())
      return fail();
    if (device < 0) device = t.get_device();
    return t.get_device() == device ? &t : fail();
  }
  // [M, cols] rows that ops._rows_contiguous passes through on the way to the fast kernels.
  const at::Tensor* rows(PyObject* o, int64_t cols) {
    const at::Tensor* t = strided(o, at::kBFloat16, 2);
    if (!t) return nullptr;
    if (M == 0) M = t->size(0);
    if (M <= 0 || t->size(0) != M || t->size(1) != cols || cols <= 1 || cols % 8 != 0 || t->stride(1) != 1) return fail();
    if (M > 1 && (t->stride(0) < cols || t->stride(0) % 8 != 0)) return fail();
    return aligned(*t) ? t : fail();
  }
  // [K, N] view of an nn.Linear weight.
  const at::Tensor* weight(PyObject* o, int64_t K, int64_t N) {
    const at::Tensor* t = strided(o, at::kBFloat16, 2);
    if (!t) return nullptr;
    return K > 1 && N > 1 && t->size(0) == K && t->size(1) == N && t->stride(0) == 1 && t->stride(1) == K ? t : fail();
  }
  const at::Tensor* mask(PyObject* o) {
    const at::Tensor* t = strided(o, at::kBool, 1);
    if (!t) return nullptr;
    return t->size(0) == M && (M <= 1 || t->stride(0) == 1) ? t : fail();
  }
  static bool aligned(const at::Tensor& t) { return reinterpret_cast<uintptr_t>(t.const_data_ptr()) % 16 == 0; }
  static int64_t ld(const at::Tensor& t) { return t.size(0) > 1 ? t.stride(0) : t.size(1); }
  bool ready() {
    if (!ok || c10::hip::current_device() != device) return false;
    stream = c10::hip::getCurrentHIPStream(device).stream();
    return true;
  }
  at::Tensor empty(const at::Tensor& like, int64_t r, int64_t c) const { return at::empty({r, c}, like.options()); }
  at::Tensor empty_weight(const at::Tensor& like, int64_t K, int64_t N) const { return at::empty_strided({K, N}, {1, K}, like.options()); }
  at::Tensor workspace(const at::Tensor& like, size_t bytes) const {
    return at::empty({(int64_t)(bytes > 16 ? bytes : 16)}, like.options().dtype(at::kByte));
  }
  // The partition the call runs with; false with a Python error set.
  bool routing(PyObject* given, PyObject* mask, Partition** r) const {
    *r = nullptr;
    if (given == Py_None && M < routed_min_rows) return true;
    PyObject* address = PyObject_CallFunction(routing_address, "OOLK", given, mask, (long long)M, (unsigned long long)(uintptr_t)stream);
    if (!address) return false;
    *r = static_cast<Partition*>(PyLong_AsVoidPtr(address));
    Py_DECREF(address);
    return !PyErr_Occurred();
  }
  // A backward whose forward left none.
  bool fill(Partition* r, const at::Tensor& mask) const {
    if (!r || r->made) return true;
    if (!run("ffnk_route", [&] {
          return lib.route(static_cast<const uint8_t*>(mask.const_data_ptr()), M, const_cast<int32_t*>(r->routing.perm),
                           const_cast<int32_t*>(r->routing.counts), stream);
        }))
      return false;
    r->made = 1;
    return true;
  }

 private:
  const at::Tensor* fail() {
    ok = false;
    return nullptr;
  }
};

int64_t size_of(PyObject* o, int64_t dim) {  // -1: no 2-D tensor
  if (!THPVariable_CheckExact(o)) return -1;
  const at::Tensor& t = THPVariable_Unpack(o);
  return t.defined() && t.dim() == 2 ? t.size(dim) : -1;
}

// (a, b1, b2, mask, routing) -> c
PyObject* linear_fwd(PyObject*, PyObject* const* p, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 5) Py_RETURN_NOTIMPLEMENTED;
  const int64_t K = size_of(p[0], 1), N = size_of(p[1], 1);
  Call c;
  const at::Tensor *a = c.rows(p[0], K), *b1 = c.weight(p[1], K, N), *b2 = c.weight(p[2], K, N), *mask = c.mask(p[3]);
  if (!c.ready()) Py_RETURN_NOTIMPLEMENTED;
  const size_t bytes = lib.workspace_bytes(FFNK_OP_LINEAR_FWD, c.M, K, N);
  if (bytes == (size_t)-1) Py_RETURN_NOTIMPLEMENTED;
  at::Tensor y = c.empty(*a, c.M, N);
  Partition* r;
  if (!c.routing(p[4], p[3], &r)) return nullptr;
  at::Tensor ws = c.workspace(*a, bytes);
  const bool fills = r && !r->made;
  if (!run("ffnk_masked_linear_fwd", [&] {
        return (fills ? lib.linear_fwd_routing : lib.linear_fwd)(
            in(*a), Call::ld(*a), in(*b1), in(*b2), 1, K, static_cast<const uint8_t*>(mask->const_data_ptr()), out(y), N, c.M, K, N,
            ws.mutable_data_ptr(), (size_t)ws.numel(), c.stream, routing_of(r));
      }))
    return nullptr;
  if (fills) r->made = 1;
  return THPVariable_Wrap(std::move(y));
  END_HANDLE_TH_ERRORS
}

// (grad, a, b1, b2, mask, routing) -> (da, db1, db2)
PyObject* linear_bwd(PyObject*, PyObject* const* p, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 6) Py_RETURN_NOTIMPLEMENTED;
  const int64_t K = size_of(p[1], 1), N = size_of(p[2], 1);
  Call c;
  const at::Tensor *g = c.rows(p[0], N), *a = c.rows(p[1], K), *b1 = c.weight(p[2], K, N), *b2 = c.weight(p[3], K, N), *mask = c.mask(p[4]);
  if (!c.ready()) Py_RETURN_NOTIMPLEMENTED;
  const size_t bytes = lib.workspace_bytes(FFNK_OP_LINEAR_BWD, c.M, K, N);
  if (bytes == (size_t)-1) Py_RETURN_NOTIMPLEMENTED;
  at::Tensor da = c.empty(*a, c.M, K), d1 = c.empty_weight(*b1, K, N), d2 = c.empty_weight(*b2, K, N);
  Partition* r;
  if (!c.routing(p[5], p[4], &r)) return nullptr;
  at::Tensor ws = c.workspace(*a, bytes);
  if (!c.fill(r, *mask)) return nullptr;
  if (!run("ffnk_masked_linear_bwd", [&] {
        return lib.linear_bwd(in(*g), Call::ld(*g), in(*a), Call::ld(*a), in(*b1), in(*b2), 1, K,
                              static_cast<const uint8_t*>(mask->const_data_ptr()), out(da), K, out(d1), out(d2), 1, K, c.M, K, N,
                              ws.mutable_data_ptr(), (size_t)ws.numel(), c.stream, routing_of(r));
      }))
    return nullptr;
  return Py_BuildValue("NNN", THPVariable_Wrap(std::move(da)), THPVariable_Wrap(std::move(d1)), THPVariable_Wrap(std::move(d2)));
  END_HANDLE_TH_ERRORS
}

// (a, w1, w2, w3, u1, u2, u3, mask, save_pre, routing) -> out, or (out, pre or None) with save_pre
PyObject* ffn_fwd(PyObject*, PyObject* const* p, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 10) Py_RETURN_NOTIMPLEMENTED;
  const int64_t d = size_of(p[0], 1), h = size_of(p[1], 1);
  Call c;
  const at::Tensor* a = c.rows(p[0], d);
  const at::Tensor* w[6];
  for (int i = 0; i < 6; ++i) w[i] = i % 3 == 1 ? c.weight(p[1 + i], h, d) : c.weight(p[1 + i], d, h);
  const at::Tensor* mask = c.mask(p[7]);
  if (!c.ready()) Py_RETURN_NOTIMPLEMENTED;
  const bool save = p[8] == Py_True;
  const size_t bytes = lib.workspace_bytes(FFNK_OP_FFN_FWD, c.M, d, h);
  if (bytes == (size_t)-1) Py_RETURN_NOTIMPLEMENTED;
  at::Tensor y = c.empty(*a, c.M, d), pre;
  if (save && lib.can_save(c.M, d, h)) pre = c.empty(*a, c.M, 2 * h);
  Partition* r;
  if (!c.routing(p[9], p[7], &r)) return nullptr;
  at::Tensor ws = c.workspace(*a, bytes);
  const bool fills = r && !r->made;
  if (!run("ffnk_masked_ffn_fwd", [&] {
        return (fills ? lib.ffn_fwd_routing : lib.ffn_fwd)(
            in(*a), Call::ld(*a), in(*w[0]), in(*w[2]), in(*w[3]), in(*w[5]), 1, d, in(*w[1]), in(*w[4]), 1, h,
            static_cast<const uint8_t*>(mask->const_data_ptr()), out(y), d, pre.defined() ? out(pre) : nullptr,
            pre.defined() ? 2 * h : 0, c.M, d, h, ws.mutable_data_ptr(), (size_t)ws.numel(), c.stream, routing_of(r));
      }))
    return nullptr;
  if (fills) r->made = 1;
  if (!save) return THPVariable_Wrap(std::move(y));
  return Py_BuildValue("NN", THPVariable_Wrap(std::move(y)), pre.defined() ? THPVariable_Wrap(std::move(pre)) : Py_NewRef(Py_None));
  END_HANDLE_TH_ERRORS
}

// (grad, a, w1, w2, w3, u1, u2, u3, mask, pre or None, routing) -> (da, dw1, dw2, dw3, du1, du2, du3)
PyObject* ffn_bwd(PyObject*, PyObject* const* p, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 11) Py_RETURN_NOTIMPLEMENTED;
  const int64_t d = size_of(p[1], 1), h = size_of(p[2], 1);
  if (h % 8 != 0) Py_RETURN_NOTIMPLEMENTED;
  Call c;
  const at::Tensor *g = c.rows(p[0], d), *a = c.rows(p[1], d);
  const at::Tensor* w[6];
  for (int i = 0; i < 6; ++i) {
    w[i] = i % 3 == 1 ? c.weight(p[2 + i], h, d) : c.weight(p[2 + i], d, h);
    if (w[i] && !Call::aligned(*w[i])) c.ok = false;  // (the lean workspace is for aligned weights)
  }
  const at::Tensor* mask = c.mask(p[8]);
  const at::Tensor* pre = p[9] == Py_None ? nullptr : c.strided(p[9], at::kBFloat16, 2);
  if (pre && (pre->size(0) != c.M || pre->size(1) != 2 * h || pre->stride(1) != 1)) c.ok = false;
  if (!c.ready()) Py_RETURN_NOTIMPLEMENTED;
  at::Tensor da = c.empty(*a, c.M, d), dw[6];
  for (int i = 0; i < 6; ++i) dw[i] = i % 3 == 1 ? c.empty_weight(*w[i], h, d) : c.empty_weight(*w[i], d, h);
  // ops.py sizes this one: what it needs depends on the layout, and the rule is there.
  THPObjectPtr space(PyObject_CallFunction(ffn_bwd_workspace, "OLLL", p[1], (long long)d, (long long)h, (long long)Call::ld(*g)));
  if (!space) return nullptr;
  const at::Tensor& ws = THPVariable_Unpack(space.get());
  Partition* r;
  if (!c.routing(p[10], p[8], &r)) return nullptr;
  if (!c.fill(r, *mask)) return nullptr;
  if (!run("ffnk_masked_ffn_bwd", [&] {
        return lib.ffn_bwd(in(*g), Call::ld(*g), in(*a), Call::ld(*a), in(*w[0]), in(*w[2]), in(*w[3]), in(*w[5]), 1, d, in(*w[1]),
                           in(*w[4]), 1, h, static_cast<const uint8_t*>(mask->const_data_ptr()), pre ? in(*pre) : nullptr,
                           pre ? Call::ld(*pre) : 0, out(da), d, out(dw[0]), out(dw[2]), out(dw[3]), out(dw[5]), 1, d, out(dw[1]),
                           out(dw[4]), 1, h, c.M, d, h, ws.mutable_data_ptr(), (size_t)ws.numel(), c.stream, routing_of(r));
      }))
    return nullptr;
  PyObject* grads = PyTuple_New(7);
  if (!grads) return nullptr;
  PyTuple_SET_ITEM(grads, 0, THPVariable_Wrap(std::move(da)));
  for (int i = 0; i < 6; ++i) PyTuple_SET_ITEM(grads, 1 + i, THPVariable_Wrap(std::move(dw[i])));
  return grads;
  END_HANDLE_TH_ERRORS
}

// (addresses of the library's functions in Library's order, routing_address, ffn_bwd_workspace, check, routed_min_rows)
PyObject* bind(PyObject*, PyObject* args) {
  PyObject *addresses, *route, *space, *raise;
  long long rows;
  if (!PyArg_ParseTuple(args, "O!OOOL", &PyTuple_Type, &addresses, &route, &space, &raise, &rows)) return nullptr;
  constexpr Py_ssize_t kFunctions = sizeof(Library) / sizeof(void*);
  if (PyTuple_GET_SIZE(addresses) != kFunctions) {
    PyErr_SetString(PyExc_ValueError, "bind: wrong number of functions");
    return nullptr;
  }
  void* f[kFunctions];
  for (Py_ssize_t i = 0; i < kFunctions; ++i) {
    f[i] = PyLong_AsVoidPtr(PyTuple_GET_ITEM(addresses, i));
    if (!f[i]) return nullptr;
  }
  memcpy(&lib, f, sizeof(lib));
  Py_INCREF(route);
  Py_INCREF(space);
  Py_INCREF(raise);
  Py_XSETREF(routing_address, route);
  Py_XSETREF(ffn_bwd_workspace, space);
  Py_XSETREF(check, raise);
  routed_min_rows = rows;
  Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"bind", bind, METH_VARARGS, nullptr},
    {"linear_fwd", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(linear_fwd)), METH_FASTCALL, nullptr},
    {"linear_bwd", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(linear_bwd)), METH_FASTCALL, nullptr},
    {"ffn_fwd", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(ffn_fwd)), METH_FASTCALL, nullptr},
    {"ffn_bwd", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(ffn_bwd)), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_call", nullptr, -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__call() { return PyModule_Create(&module); }
