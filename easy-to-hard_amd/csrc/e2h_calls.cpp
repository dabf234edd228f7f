// Calls of a quantized linear on plain tensors, host side: what ops._int4_mm_impl and ops._int8_mm_impl do for up to 1023 rows, in one native call.
//
// A call of a small linear through Python is bound by the host.  4096 x 4096 at one row, group size 128: the kernel takes 7.0 us, and the checks, the allocation, the workspace's lookup
// and the ctypes call of the Python path together with nn.Module's part 11.6; from here 7.3 (see WeightOnlyInt4Linear.forward).  Anything out of the ordinary -- tensor subclasses
// and wrappers, modes, traces, other types, strides, devices or shapes, captures, a workspace that is not there yet -- returns None, and the Python path takes the call or
// raises its error, and so it does where an entry point refuses its arguments.  A launch that failed is reported from here: asked once more, the
// runtime may take it, over whatever of a call of several launches has begun.
//
// The functions take (x, weight, scales, .., out_features, ..) and return a new tensor or None.
#include <Python.h>

#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>

#include <cstdint>

namespace {

typedef int (*Int4Mm)(const void *, const void *, const void *, void *, int64_t, int64_t, int64_t, int, int, void *, int64_t, void *);
typedef int (*Int8Mm)(const void *, const void *, const void *, void *, int64_t, int64_t, int64_t, void *, int64_t, void *);
typedef int (*Int4Rows)(const void *, const void *, const void *, void *, int, void *, void *, int64_t, int64_t, int64_t, int, int, void *);
typedef int (*Int4RowsSlices)(int64_t, int64_t, int64_t, int, int);
typedef int (*Capturing)(void *);

Int4Mm int4_mm_entry = nullptr;
Int8Mm int8_mm_entry = nullptr;
Int4Rows int4_rows_entry = nullptr;
Int4RowsSlices int4_rows_slices_entry = nullptr;
Capturing capturing_entry = nullptr;
PyObject *workspaces = nullptr;  // ops._workspaces: (device index, stream) -> tensor
PyObject *check = nullptr;       // _lib.check: raises what a status stands for

constexpr int64_t kMostRows = 1023;  // larger calls may use memory of their own

// E2H_ERR_LAUNCH and E2H_ERR_NO_DEVICE of e2h_quant.h: what does not follow from the arguments
bool failed(int status) { return status == -6 || status == -7; }

// a tensor of this device and type whose elements lie as its shape says, with nothing that follows what happens to it
bool plain(const at::Tensor &t, c10::DeviceIndex device, at::ScalarType type) {
  static const c10::DispatchKeySet kept = c10::DispatchKeySet({c10::DispatchKey::CUDA, c10::DispatchKey::ADInplaceOrView, c10::DispatchKey::AutogradCUDA, c10::DispatchKey::AutocastCUDA});
  static const c10::DispatchKeySet left(c10::BackendComponent::CUDABit);  // a difference of key sets keeps the backend
  return t.defined() && t.is_cuda() && t.get_device() == device && t.scalar_type() == type && t.key_set() - kept == left && t.is_contiguous();
}

bool watched() {
  return at::impl::torch_function_mode_enabled() || c10::impl::TorchDispatchModeTLS::any_modes_set() || torch::jit::tracer::isTracing();
}

// the workspace's address and size for launches on the stream; false: there is none yet, or the stream records a graph
bool workspace_of(c10::DeviceIndex device, void *stream, void **ptr, int64_t *bytes) {
  if (capturing_entry(stream) != 0) return false;
  PyObject *key = Py_BuildValue("(iK)", static_cast<int>(device), static_cast<unsigned long long>(reinterpret_cast<uintptr_t>(stream)));
  if (!key) {
    PyErr_Clear();
    return false;
  }
  PyObject *ws = PyDict_GetItemWithError(workspaces, key);  // borrowed
  Py_DECREF(key);
  if (!ws || !THPVariable_Check(ws)) {
    PyErr_Clear();
    return false;
  }
  const at::Tensor &t = THPVariable_Unpack(ws);
  *ptr = t.data_ptr();
  *bytes = t.numel();
  return true;
}

// [.., n] beside x [.., k]
at::Tensor result_for(const at::Tensor &x, int64_t n) {
  c10::SmallVector<int64_t, 5> sizes(x.sizes().begin(), x.sizes().end());
  sizes.back() = n;
  return at::empty(sizes, x.options());
}

template <class Launch>
PyObject *run(const char *entry, const at::Tensor &x, int64_t n, c10::DeviceIndex device, Launch launch) {
  void *const stream = c10::hip::getCurrentHIPStream(device).stream();
  void *ws = nullptr;
  int64_t ws_bytes = 0;
  if (!workspace_of(device, stream, &ws, &ws_bytes)) Py_RETURN_NONE;
  at::Tensor y = result_for(x, n);
  int rc;
  Py_BEGIN_ALLOW_THREADS  // a full queue makes the launch wait
  rc = launch(y.data_ptr(), ws, ws_bytes, stream);
  Py_END_ALLOW_THREADS
  if (failed(rc)) {
    Py_XDECREF(PyObject_CallFunction(check, "is", rc, entry));
    return nullptr;
  }
  if (rc != 0) Py_RETURN_NONE;  // the Python path meets the same status and raises it
  return THPVariable_Wrap(std::move(y));
}

struct Int4Call {
  c10::DeviceIndex device;
  int64_t m, n, k, g;
};

// the sizes of x beside packed weights with inner_k_tiles 8; false: not for here
bool int4_call(const at::Tensor &x, const at::Tensor &w, const at::Tensor &sz, int64_t g, int64_t out, Int4Call *c) {
  if (!x.defined() || !x.is_cuda()) return false;
  c->device = x.get_device();
  if (c->device != c10::hip::current_device() || !plain(x, c->device, at::kBFloat16) || !plain(w, c->device, at::kInt) || !plain(sz, c->device, at::kBFloat16)) return false;
  if (x.dim() < 1 || w.dim() != 4 || sz.dim() != 3 || w.size(2) != 32 || w.size(3) != 4) return false;
  c->n = w.size(0) * 8, c->k = w.size(1) * 128, c->m = c->k > 0 ? x.numel() / c->k : 0, c->g = g;
  if (x.size(-1) != c->k || c->n != out || c->m < 1 || c->m > kMostRows || (g != 32 && g != 64 && g != 128 && g != 256) || c->k % g != 0) return false;
  return sz.size(0) == c->k / g && sz.size(1) == c->n && sz.size(2) == 2;
}

// (x, packed, scales_and_zeros, groupsize, out_features); inner_k_tiles 8
PyObject *int4_linear(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  if (nargs != 5 || !int4_mm_entry || !THPVariable_CheckExact(args[0]) || !THPVariable_CheckExact(args[1]) || !THPVariable_CheckExact(args[2]) || watched()) Py_RETURN_NONE;
  const int64_t g = PyLong_AsLongLong(args[3]), out = PyLong_AsLongLong(args[4]);
  if (PyErr_Occurred()) {
    PyErr_Clear();
    Py_RETURN_NONE;
  }
  const at::Tensor &x = THPVariable_Unpack(args[0]), &w = THPVariable_Unpack(args[1]), &sz = THPVariable_Unpack(args[2]);
  Int4Call c;
  if (!int4_call(x, w, sz, g, out, &c)) Py_RETURN_NONE;
  return run("e2h_int4_mm", x, c.n, c.device, [&](void *y, void *ws, int64_t ws_bytes, void *stream) {
    return int4_mm_entry(x.data_ptr(), w.data_ptr(), sz.data_ptr(), y, c.m, c.n, c.k, static_cast<int>(g), 8, ws, ws_bytes, stream);
  });
  END_HANDLE_TH_ERRORS
}

// (x, packed, scales_and_zeros, groupsize, out_features, sums or None, defer): e2h_int4_mm_rows, where it takes the call.  sums: e2h_add_rmsnorm_sums' of x.  defer: where K is shared, the slices'
// sums [slices, m, n] in the result's place.
PyObject *int4_rows(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  if (nargs != 7 || !int4_rows_entry || !THPVariable_CheckExact(args[0]) || !THPVariable_CheckExact(args[1]) || !THPVariable_CheckExact(args[2]) ||
      (args[5] != Py_None && !THPVariable_CheckExact(args[5])) || watched())
    Py_RETURN_NONE;
  const int64_t g = PyLong_AsLongLong(args[3]), out = PyLong_AsLongLong(args[4]);
  const bool defer = args[6] == Py_True, there = args[5] != Py_None;
  if (PyErr_Occurred()) {
    PyErr_Clear();
    Py_RETURN_NONE;
  }
  const at::Tensor &x = THPVariable_Unpack(args[0]), &w = THPVariable_Unpack(args[1]), &sz = THPVariable_Unpack(args[2]);
  Int4Call c;
  if (!int4_call(x, w, sz, g, out, &c)) Py_RETURN_NONE;
  const int slices = int4_rows_slices_entry(c.m, c.n, c.k, static_cast<int>(g), 8);
  void *const stream = c10::hip::getCurrentHIPStream(c.device).stream();
  if (slices < 1 || capturing_entry(stream) != 0) Py_RETURN_NONE;
  const int64_t groups = c.k / (g < 128 ? g : 128), stride = (c.m + 63) / 64 * 64;
  const auto floats = x.options().dtype(at::kFloat);
  at::Tensor sums, partials, y;
  if (there) {
    sums = THPVariable_Unpack(args[5]);
    if (!plain(sums, c.device, at::kFloat) || sums.dim() != 2 || sums.size(0) != groups || sums.size(1) != stride) Py_RETURN_NONE;
  }
  try {
    if (!there) sums = at::empty({groups, stride}, floats);
    if (slices > 1) partials = at::empty({slices, c.m, c.n}, floats);
  } catch (const c10::OutOfMemoryError &) {
    Py_RETURN_NONE;  // the calls without this have a workspace for both
  }
  if (slices == 1 || !defer) y = result_for(x, c.n);
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = int4_rows_entry(x.data_ptr(), w.data_ptr(), sz.data_ptr(), sums.data_ptr(), there, y.defined() ? y.data_ptr() : nullptr, partials.defined() ? partials.data_ptr() : nullptr, c.m, c.n,
                       c.k, static_cast<int>(g), 8, stream);
  Py_END_ALLOW_THREADS
  if (failed(rc)) {
    Py_XDECREF(PyObject_CallFunction(check, "is", rc, "e2h_int4_mm_rows"));
    return nullptr;
  }
  if (rc != 0) Py_RETURN_NONE;
  return THPVariable_Wrap(std::move(y.defined() ? y : partials));
  END_HANDLE_TH_ERRORS
}

// (x, q, scales, out_features)
PyObject *int8_linear(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  if (nargs != 4 || !int8_mm_entry || !THPVariable_CheckExact(args[0]) || !THPVariable_CheckExact(args[1]) || !THPVariable_CheckExact(args[2]) || watched()) Py_RETURN_NONE;
  const int64_t out = PyLong_AsLongLong(args[3]);
  if (PyErr_Occurred()) {
    PyErr_Clear();
    Py_RETURN_NONE;
  }
  const at::Tensor &x = THPVariable_Unpack(args[0]), &q = THPVariable_Unpack(args[1]), &scales = THPVariable_Unpack(args[2]);
  if (!x.defined() || !x.is_cuda()) Py_RETURN_NONE;
  const c10::DeviceIndex device = x.get_device();
  if (device != c10::hip::current_device() || !plain(x, device, at::kBFloat16) || !plain(q, device, at::kChar) || !plain(scales, device, at::kBFloat16)) Py_RETURN_NONE;
  if (x.dim() < 1 || q.dim() != 2 || scales.dim() != 1) Py_RETURN_NONE;
  const int64_t n = q.size(0), k = q.size(1), m = k > 0 ? x.numel() / k : 0;
  if (x.size(-1) != k || n != out || n < 1 || m < 1 || m > kMostRows || scales.size(0) != n) Py_RETURN_NONE;
  return run("e2h_int8_mm", x, n, device, [&](void *y, void *ws, int64_t ws_bytes, void *stream) {
    return int8_mm_entry(x.data_ptr(), q.data_ptr(), scales.data_ptr(), y, m, n, k, ws, ws_bytes, stream);
  });
  END_HANDLE_TH_ERRORS
}

// bind(address of e2h_int4_mm, of e2h_int8_mm, of e2h_stream_capturing, ops._workspaces, _lib.check)
PyObject *bind(PyObject *, PyObject *args) {
  unsigned long long int4 = 0, int8 = 0, capturing = 0;
  PyObject *dict = nullptr, *raises = nullptr;
  if (!PyArg_ParseTuple(args, "KKKO!O", &int4, &int8, &capturing, &PyDict_Type, &dict, &raises)) return nullptr;
  Py_INCREF(dict);
  Py_INCREF(raises);
  Py_XDECREF(workspaces);
  Py_XDECREF(check);
  workspaces = dict;
  check = raises;
  int4_mm_entry = reinterpret_cast<Int4Mm>(static_cast<uintptr_t>(int4));
  int8_mm_entry = reinterpret_cast<Int8Mm>(static_cast<uintptr_t>(int8));
  capturing_entry = reinterpret_cast<Capturing>(static_cast<uintptr_t>(capturing));
  Py_RETURN_NONE;
}

// bind_rows(address of e2h_int4_mm_rows, of e2h_int4_mm_rows_slices)
PyObject *bind_rows(PyObject *, PyObject *args) {
  unsigned long long rows = 0, slices = 0;
  if (!PyArg_ParseTuple(args, "KK", &rows, &slices)) return nullptr;
  int4_rows_entry = reinterpret_cast<Int4Rows>(static_cast<uintptr_t>(rows));
  int4_rows_slices_entry = reinterpret_cast<Int4RowsSlices>(static_cast<uintptr_t>(slices));
  Py_RETURN_NONE;
}

PyMethodDef methods[] = {{"int4_linear", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(int4_linear)), METH_FASTCALL, nullptr},
                         {"int8_linear", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(int8_linear)), METH_FASTCALL, nullptr},
                         {"int4_rows", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(int4_rows)), METH_FASTCALL, nullptr},
                         {"bind", bind, METH_VARARGS, nullptr},
                         {"bind_rows", bind_rows, METH_VARARGS, nullptr},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_calls", nullptr, -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__calls(void) {
  PyObject *m = PyModule_Create(&module);
  if (m && PyModule_AddStringConstant(m, "torch_version", E2H_TORCH_VERSION) != 0) Py_CLEAR(m);  // compared before anything here touches a tensor
  return m;
}
