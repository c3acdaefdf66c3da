// CPython entry points of the calls a decode loop makes per layer and step (include/espetero_attn.h), arguments in the
// header's order without the error buffer: records as instances of their own ctypes classes (abi.AttnParams, PrepParams,
// GateParams), device memory as torch tensors or None, the stream as an integer. Anything else is refused before the library
// is called: it would read another record's bytes, or a number, as an address. A failing call raises abi.EspError.
//
// Why native: a decode step of one short sequence is 8 us of GPU work behind two launches, and the ctypes form of the
// same call - an error buffer, twenty pointer objects, a Stream object - cost the host about as much as the launches
// themselves (10.6 us a step of one 1024-key sequence; in this form 8.3, the GPU being the slower side). The conversions below take one pass over the arguments.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <cstdint>
#include <cstdio>
#include <tuple>
#include <type_traits>
#include <utility>

#include "../../include/espetero_attn.h"

namespace {

PyObject* g_data_ptr;  // interned "data_ptr"
PyObject* g_error;     // abi.EspError
// abi's classes of the parameter records
PyTypeObject *g_attn_params, *g_prep_params, *g_gate_params;

// A structure's bytes, held until the call has returned.
struct Record {
  Py_buffer view{};
  ~Record() {
    if (view.obj) PyBuffer_Release(&view);
  }
};

// The address of a tensor (of whatever has a data_ptr method); None: a null pointer.
bool address(PyObject* o, void*& out) {
  if (o == Py_None) {
    out = nullptr;
    return true;
  }
  PyObject* v = PyObject_VectorcallMethod(g_data_ptr, &o, 1 | PY_VECTORCALL_ARGUMENTS_OFFSET, nullptr);
  if (!v) return false;
  out = PyLong_AsVoidPtr(v);
  Py_DECREF(v);
  return !(out == nullptr && PyErr_Occurred());
}

template <typename T>
PyTypeObject* record_class() {
  if constexpr (std::is_same_v<T, const esp_attn_params*>) return g_attn_params;
  else if constexpr (std::is_same_v<T, const esp_prep_params*>) return g_prep_params;
  else if constexpr (std::is_same_v<T, const esp_gate_params*>) return g_gate_params;
  else return nullptr;
}

template <typename T>
constexpr bool is_params = std::is_same_v<T, const esp_attn_params*> || std::is_same_v<T, const esp_prep_params*> ||
                           std::is_same_v<T, const esp_gate_params*>;

// stream: the call's last argument, a hipStream_t as an integer.
template <bool stream, typename T>
bool convert(PyObject* o, T& out, Record& rec) {
  if constexpr (is_params<T>) {
    PyTypeObject* const cls = record_class<T>();
    if (!PyObject_TypeCheck(o, cls)) {
      PyErr_Format(PyExc_TypeError, "%s expected, not %s", cls->tp_name, Py_TYPE(o)->tp_name);
      return false;
    }
    if (PyObject_GetBuffer(o, &rec.view, PyBUF_SIMPLE) != 0) return false;
    if (size_t(rec.view.len) < sizeof(std::remove_pointer_t<T>)) {
      PyErr_SetString(PyExc_ValueError, "parameter record too small");
      return false;
    }
    out = static_cast<T>(rec.view.buf);
    return true;
  } else if constexpr (stream) {
    out = static_cast<T>(PyLong_AsVoidPtr(o));
    return !(out == nullptr && PyErr_Occurred());
  } else if constexpr (std::is_pointer_v<T>) {
    void* p = nullptr;
    if (!address(o, p)) return false;
    out = static_cast<T>(p);
    return true;
  } else if constexpr (std::is_signed_v<T>) {
    const long v = PyLong_AsLong(o);
    if (v == -1 && PyErr_Occurred()) return false;
    if (v < INT32_MIN || v > INT32_MAX) {
      PyErr_SetString(PyExc_OverflowError, "a count or size does not fit 32 bits");
      return false;
    }
    out = T(v);
    return true;
  } else {  // any integer, numpy's among them
    out = T(PyLong_AsUnsignedLongLongMask(o));
    return !(out == T(-1) && PyErr_Occurred());
  }
}

// The function's parameters less the last two (the error buffer and its length).
template <auto Fn, typename... A, size_t... I>
PyObject* run(int (*)(A...), std::index_sequence<I...>, PyObject* const* args, Py_ssize_t n) {
  if (n != Py_ssize_t(sizeof...(I))) return PyErr_Format(PyExc_TypeError, "%zd arguments, %zd expected", n, Py_ssize_t(sizeof...(I)));
  using All = std::tuple<A...>;
  std::tuple<std::tuple_element_t<I, All>...> v{};
  Record rec[sizeof...(I)];
  if (!(convert<I + 1 == sizeof...(I)>(args[I], std::get<I>(v), rec[I]) && ...)) return nullptr;
  char err[512];
  err[0] = 0;
  int rc;
  Py_BEGIN_ALLOW_THREADS;
  rc = Fn(std::get<I>(v)..., err, sizeof err);
  Py_END_ALLOW_THREADS;
  if (rc == ESP_OK) Py_RETURN_NONE;
  return PyErr_Format(g_error, "esp error %d: %s", rc, err);
}

template <typename... A>
constexpr size_t arity(int (*)(A...)) {
  return sizeof...(A);
}

template <auto Fn>
PyObject* call(PyObject*, PyObject* const* args, Py_ssize_t n) {
  return run<Fn>(Fn, std::make_index_sequence<arity(Fn) - 2>{}, args, n);
}

#define ESP_CALL(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&call<esp_##name>)), METH_FASTCALL, nullptr}
PyMethodDef g_methods[] = {ESP_CALL(attn_forward),   ESP_CALL(attn_forward_static), ESP_CALL(attn_decode_fused), ESP_CALL(attn_prep),
                           ESP_CALL(attn_combine),   ESP_CALL(head_gate),           ESP_CALL(kv_save),           ESP_CALL(kv_copy_blocks),
                           ESP_CALL(kv_export_blocks), ESP_CALL(kv_import_blocks),  ESP_CALL(chain_advance),     {nullptr, nullptr, 0, nullptr}};
PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_calls", nullptr, -1, g_methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__calls() {
  PyObject* abi = PyImport_ImportModule("espetero_amd.abi");
  if (!abi) return nullptr;
  g_error = PyObject_GetAttrString(abi, "EspError");
  g_attn_params = reinterpret_cast<PyTypeObject*>(PyObject_GetAttrString(abi, "AttnParams"));
  g_prep_params = reinterpret_cast<PyTypeObject*>(PyObject_GetAttrString(abi, "PrepParams"));
  g_gate_params = reinterpret_cast<PyTypeObject*>(PyObject_GetAttrString(abi, "GateParams"));
  PyObject* version = PyObject_GetAttrString(abi, "ESP_ABI_VERSION");
  Py_DECREF(abi);
  g_data_ptr = PyUnicode_InternFromString("data_ptr");
  if (!g_error || !g_attn_params || !g_prep_params || !g_gate_params || !version || !g_data_ptr) {
    Py_XDECREF(version);
    return nullptr;
  }
  // The library that was loaded, this file and abi's records have to be of one version: as abi.attn_lib() checks for ctypes.
  const long want = PyLong_AsLong(version);
  Py_DECREF(version);
  if (want == -1 && PyErr_Occurred()) return nullptr;
  if (esp_attn_abi_version() != want || want != ESP_ABI_VERSION) {
    PyErr_SetString(g_error, "libespetero_attn.so: ABI version mismatch");
    return nullptr;
  }
  return PyModule_Create(&g_module);
}
