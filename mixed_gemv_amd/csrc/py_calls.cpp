// The device entry points as CPython calls.
//
// A decode step is a chain of launches of a few microseconds each, so the way from a Python call to the
// launch is part of what a product costs: through ctypes and torch's Python objects it took 8.8 us a call
// (13 argument conversions, 5 tensors asked for address, device and contiguity, and torch.cuda.current_stream(),
// 2.8 us of it), longer than the kernel of a 4096x4096 product runs (4 us).  Here the tensors are unpacked
// and the stream is found in C++.  The functions take the arguments of the wrappers in api.py by
// position and return the C-ABI's status; what they do not know -- an object that is neither a torch tensor nor an
// integer, a failed check -- is handed to the Python helper that words the error or finds the address.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include "mixed_gemv.h"

namespace {

PyObject* g_dev_address = nullptr;   // api._dev_address: address of an object this file does not know, or the error
PyObject* g_is_bf16 = nullptr;       // api._is_bf16
PyObject* g_stream_address = nullptr;  // api._stream_address

struct Failed {};  // a Python exception is set

const at::Tensor* as_tensor(PyObject* o) { return THPVariable_Check(o) ? &THPVariable_Unpack(o) : nullptr; }

uintptr_t address_from_python(PyObject* helper, PyObject* o) {
  PyObject* r = PyObject_CallOneArg(helper, o);
  if (r == nullptr) throw Failed{};
  const uintptr_t v = (uintptr_t)PyLong_AsVoidPtr(r);
  Py_DECREF(r);
  if (v == 0 && PyErr_Occurred()) throw Failed{};
  return v;
}

// None, an integer address, or a contiguous GPU tensor.
template <typename T>
T* device_pointer(PyObject* o) {
  if (o == Py_None) return nullptr;
  if (const at::Tensor* t = as_tensor(o)) {
    if (t->layout() == c10::kStrided && t->is_cuda() && t->is_contiguous()) return static_cast<T*>(t->data_ptr());
  }
  return reinterpret_cast<T*>(address_from_python(g_dev_address, o));
}

int64_t integer(PyObject* o) {
  int64_t v;
  if (PyLong_Check(o)) {
    v = PyLong_AsLongLong(o);
  } else {  // what int() takes: numpy integers, floats
    PyObject* n = PyNumber_Long(o);
    if (n == nullptr) throw Failed{};
    v = PyLong_AsLongLong(n);
    Py_DECREF(n);
  }
  if (v == -1 && PyErr_Occurred()) throw Failed{};
  return v;
}
// as a C int parameter receives it through ctypes: the low 32 bits
int small_integer(PyObject* o) { return (int)integer(o); }

// element: "f16", "bf16", or None = the type of the tensor `probe`
bool is_bf16(PyObject* element, PyObject* probe) {
  if (element == Py_None) {
    if (const at::Tensor* t = as_tensor(probe)) return t->scalar_type() == at::kBFloat16;
    if (PyLong_Check(probe) || probe == Py_None) return false;
  }
  PyObject* args[2] = {element, probe};
  PyObject* r = PyObject_Vectorcall(g_is_bf16, args, 2, nullptr);
  if (r == nullptr) throw Failed{};
  const int yes = PyObject_IsTrue(r);
  Py_DECREF(r);
  if (yes < 0) throw Failed{};
  return yes != 0;
}

// None = the current stream of the current device, as torch.cuda.current_stream() says
void* stream_of(PyObject* o) {
  if (o == Py_None) return static_cast<void*>(c10::hip::getCurrentHIPStream().stream());
  return reinterpret_cast<void*>(address_from_python(g_stream_address, o));
}

struct Strides {
  int64_t weights = 0, x = 0, scale = 0, bias = 0, y = 0;
};
Strides strides_of(PyObject* o) {
  PyObject* seq = PySequence_Fast(o, "batch_strides must be a sequence of five integers");
  if (seq == nullptr) throw Failed{};
  Strides s;
  int64_t* const into[5] = {&s.weights, &s.x, &s.scale, &s.bias, &s.y};
  try {
    if (PySequence_Fast_GET_SIZE(seq) != 5) {
      PyErr_SetString(PyExc_ValueError, "batch_strides must be five integers");
      throw Failed{};
    }
    for (int i = 0; i < 5; ++i) *into[i] = integer(PySequence_Fast_GET_ITEM(seq, i));
  } catch (...) {
    Py_DECREF(seq);
    throw;
  }
  Py_DECREF(seq);
  return s;
}

// Runs `body` (which returns a status) and turns every exception into a Python one.
template <typename Body>
PyObject* call(const char* name, Py_ssize_t got, Py_ssize_t want, Body body) {
  if (got != want) return PyErr_Format(PyExc_TypeError, "%s takes %zd arguments (%zd given)", name, want, got);
  try {
    return PyLong_FromLong(body());
  } catch (const Failed&) {
    return nullptr;
  } catch (const std::exception& e) {
    PyErr_SetString(PyExc_RuntimeError, e.what());
    return nullptr;
  }
}

// The launch itself runs without the interpreter lock: it may wait for room in the queue.
template <typename Launch>
int unlocked(Launch launch) {
  int status;
  Py_BEGIN_ALLOW_THREADS;
  status = launch();
  Py_END_ALLOW_THREADS;
  return status;
}

// ptr_A, ptr_B, ptr_scale, ptr_zero_point, ptr_C, ptr_D, B, M, N, K, group_size, quant_op, weight_bits, stream,
// batch_strides, element
PyObject* gemv(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return call("gemv", n, 16, [&] {
    const void* w = device_pointer<const void>(a[0]);
    const uint16_t* x = device_pointer<const uint16_t>(a[1]);
    const uint16_t* s = device_pointer<const uint16_t>(a[2]);
    const uint16_t* z = device_pointer<const uint16_t>(a[3]);
    const uint16_t* c = device_pointer<const uint16_t>(a[4]);
    uint16_t* y = device_pointer<uint16_t>(a[5]);
    const int batch = small_integer(a[6]), m = small_integer(a[7]), rows = small_integer(a[8]), k = small_integer(a[9]);
    const int group = small_integer(a[10]), op = small_integer(a[11]), bits = small_integer(a[12]);
    const int strided = PyObject_IsTrue(a[14]);
    if (strided < 0) throw Failed{};
    const Strides st = strided ? strides_of(a[14]) : Strides{};
    const auto entry = is_bf16(a[15], a[1]) ? mgemv_gemv_batched_bf16 : mgemv_gemv_batched;
    void* const stream = stream_of(a[13]);
    return unlocked([&] {
      return entry(w, x, s, z, c, y, batch, m, rows, k, group, op, bits, st.weights, st.x, st.scale, st.bias, st.y, stream);
    });
  });
}

// ptr_A, ptr_B, ptr_scale, ptr_zero_point, ptr_C, ptr_D, route, stack_entries, B, M, N, K, group_size, batch_strides,
// quant_op, weight_bits, stream, element
PyObject* gemv_routed(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return call("gemv_routed", n, 18, [&] {
    const void* w = device_pointer<const void>(a[0]);
    const uint16_t* x = device_pointer<const uint16_t>(a[1]);
    const uint16_t* s = device_pointer<const uint16_t>(a[2]);
    const uint16_t* z = device_pointer<const uint16_t>(a[3]);
    const uint16_t* c = device_pointer<const uint16_t>(a[4]);
    uint16_t* y = device_pointer<uint16_t>(a[5]);
    const int32_t* route = device_pointer<const int32_t>(a[6]);
    const int entries = small_integer(a[7]), batch = small_integer(a[8]), m = small_integer(a[9]);
    const int rows = small_integer(a[10]), k = small_integer(a[11]), group = small_integer(a[12]);
    const Strides st = strides_of(a[13]);
    const int op = small_integer(a[14]), bits = small_integer(a[15]);
    const auto entry = is_bf16(a[17], a[1]) ? mgemv_gemv_routed_bf16 : mgemv_gemv_routed;
    void* const stream = stream_of(a[16]);
    return unlocked([&] {
      return entry(w, x, s, z, c, y, route, entries, batch, m, rows, k, group, op, bits, st.weights, st.x, st.scale,
                   st.bias, st.y, stream);
    });
  });
}

// ptr_A, ptr_scale, ptr_zero_point, ptr_out, M, K, group_size, quant_op, weight_bits, stream, element
PyObject* dequantize(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return call("dequantize", n, 11, [&] {
    const void* w = device_pointer<const void>(a[0]);
    const uint16_t* s = device_pointer<const uint16_t>(a[1]);
    const uint16_t* z = device_pointer<const uint16_t>(a[2]);
    uint16_t* out = device_pointer<uint16_t>(a[3]);
    const int m = small_integer(a[4]), k = small_integer(a[5]), group = small_integer(a[6]);
    const int op = small_integer(a[7]), bits = small_integer(a[8]);
    const auto entry = is_bf16(a[10], a[1]) ? mgemv_dequantize_bf16 : mgemv_dequantize;
    void* const stream = stream_of(a[9]);
    return unlocked([&] { return entry(w, s, z, out, m, k, group, op, bits, stream); });
  });
}

template <PyObject* (*F)(PyObject*, PyObject* const*, Py_ssize_t)>
PyCFunction as_method() { return reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(F)); }

PyMethodDef g_methods[] = {
    {"gemv", as_method<gemv>(), METH_FASTCALL, "mgemv_gemv_batched / _bf16; returns the status"},
    {"gemv_routed", as_method<gemv_routed>(), METH_FASTCALL, "mgemv_gemv_routed / _bf16; returns the status"},
    {"dequantize", as_method<dequantize>(), METH_FASTCALL, "mgemv_dequantize / _bf16; returns the status"},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "py_calls", nullptr, -1, g_methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_py_calls() {
  PyObject* api = PyImport_ImportModule("mixed_gemv_amd.api");
  if (api == nullptr) return nullptr;
  g_dev_address = PyObject_GetAttrString(api, "_dev_address");
  g_is_bf16 = PyObject_GetAttrString(api, "_is_bf16");
  g_stream_address = PyObject_GetAttrString(api, "_stream_address");
  Py_DECREF(api);
  if (g_dev_address == nullptr || g_is_bf16 == nullptr || g_stream_address == nullptr) return nullptr;
  return PyModule_Create(&g_module);
}
