// Native half of the Python binding (l2c/__init__.py): the kernel entry points
// of include/l2c.h as functions over torch tensors, integers, floats and a
// stream, without ctypes. A wrapper's host time was about 7.6 us a call through
// ctypes (objects made for every pointer, torch's stream object), against 2 to
// 3 us for the launch itself: the small iterations and decoder steps, of one to
// six calls, waited for the host.
//
// A call converts its arguments by the C function's own parameter types:
//   pointer        None, or an object with is_cuda (true) and data_ptr()
//   int, size_t,   Python integers in range
//   long long
//   float          Python floats and integers
//   hipStream_t    None (torch's current stream on the current device), an
//                  integer, or an object with cuda_stream
// Arguments of any other form go to the Python fallback, which converts them (or
// raises) as ctypes does. The GIL is released around the C call, as ctypes does.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <climits>
#include <cstdint>
#include <tuple>
#include <type_traits>
#include <utility>

#include "l2c.h"

namespace {

PyObject *g_raw_stream = nullptr;  // torch's raw current stream of a device index
PyObject *g_fallback = nullptr;    // fallback(name, *args) -> return code
PyObject *g_is_cuda = nullptr, *g_data_ptr = nullptr, *g_cuda_stream = nullptr;

// Each converter returns false, with no Python error set, for an argument it
// does not take.
bool no_error() {
  PyErr_Clear();
  return false;
}

bool to_address(PyObject *o, uintptr_t *v) {
  if (!PyLong_Check(o)) return false;
  const unsigned long long u = PyLong_AsUnsignedLongLong(o);
  if (u == static_cast<unsigned long long>(-1) && PyErr_Occurred()) return no_error();
  *v = static_cast<uintptr_t>(u);
  return true;
}

bool attribute_address(PyObject *o, uintptr_t *v) {  // takes the reference to o
  if (!o) return no_error();
  const bool ok = to_address(o, v);
  Py_DECREF(o);
  return ok;
}

template <typename T>
bool convert(PyObject *o, T **v) {
  *v = nullptr;
  if (o == Py_None) return true;
  PyObject *cuda = PyObject_GetAttr(o, g_is_cuda);
  if (!cuda) return no_error();
  const bool on_gpu = cuda == Py_True;
  Py_DECREF(cuda);
  uintptr_t p = 0;
  if (!on_gpu || !attribute_address(PyObject_CallMethodNoArgs(o, g_data_ptr), &p)) return false;
  *v = reinterpret_cast<T *>(p);
  return true;
}

bool convert(PyObject *o, hipStream_t *v) {
  uintptr_t p = 0;
  if (o == Py_None) {
    int device = 0;
    if (hipGetDevice(&device) != hipSuccess) return false;
    PyObject *index = PyLong_FromLong(device);
    if (!index) return no_error();
    PyObject *raw = PyObject_CallOneArg(g_raw_stream, index);
    Py_DECREF(index);
    if (!attribute_address(raw, &p)) return false;
  } else if (PyLong_Check(o)) {
    if (!to_address(o, &p)) return false;
  } else if (!attribute_address(PyObject_GetAttr(o, g_cuda_stream), &p)) {
    return false;
  }
  *v = reinterpret_cast<hipStream_t>(p);
  return true;
}

bool convert(PyObject *o, int *v) {
  if (!PyLong_Check(o)) return false;
  int overflow = 0;
  const long n = PyLong_AsLongAndOverflow(o, &overflow);
  if (overflow || n < INT_MIN || n > INT_MAX) return false;
  *v = static_cast<int>(n);
  return true;
}

bool convert(PyObject *o, long long *v) {
  if (!PyLong_Check(o)) return false;
  int overflow = 0;
  *v = PyLong_AsLongLongAndOverflow(o, &overflow);
  return !overflow;
}

bool convert(PyObject *o, size_t *v) {
  uintptr_t u = 0;
  if (!to_address(o, &u)) return false;
  *v = u;
  return true;
}

bool convert(PyObject *o, float *v) {
  if (!PyFloat_CheckExact(o)) return false;
  *v = static_cast<float>(PyFloat_AS_DOUBLE(o));
  return true;
}

template <typename... P, size_t... I>
bool run(int (*fn)(P...), PyObject *const *args, std::index_sequence<I...>, int *code) {
  std::tuple<P...> v;
  if (!(convert(args[I], &std::get<I>(v)) && ...)) return false;
  Py_BEGIN_ALLOW_THREADS;
  *code = fn(std::get<I>(v)...);
  Py_END_ALLOW_THREADS;
  return true;
}

template <typename... P>
bool run(int (*fn)(P...), PyObject *const *args, Py_ssize_t n, int *code) {
  return n == static_cast<Py_ssize_t>(sizeof...(P)) && run(fn, args, std::index_sequence_for<P...>(), code);
}

PyObject *fall_back(const char *name, PyObject *const *args, Py_ssize_t n) {
  PyObject *all = PyTuple_New(n + 1);
  if (!all) return nullptr;
  PyObject *text = PyUnicode_FromString(name);
  if (!text) {
    Py_DECREF(all);
    return nullptr;
  }
  PyTuple_SET_ITEM(all, 0, text);
  for (Py_ssize_t i = 0; i < n; ++i) {
    Py_INCREF(args[i]);
    PyTuple_SET_ITEM(all, i + 1, args[i]);
  }
  PyObject *result = PyObject_CallObject(g_fallback, all);
  Py_DECREF(all);
  return result;
}

// Python function of one entry point: its return code.
#define L2C_ENTRY(NAME)                                                           \
  PyObject *py_##NAME(PyObject *, PyObject *const *args, Py_ssize_t n) {          \
    int code = 0;                                                                 \
    if (!g_fallback) {                                                            \
      PyErr_SetString(PyExc_RuntimeError, "l2c_native is not initialised");       \
      return nullptr;                                                             \
    }                                                                             \
    if (!run(l2c_##NAME, args, n, &code)) return fall_back("l2c_" #NAME, args, n); \
    return PyLong_FromLong(code);                                                 \
  }
#define L2C_ENTRIES(X)                                                                                          \
  X(rmsnorm) X(softmax) X(matvec) X(fused) X(matmul) X(matmul_q) X(matmul_qs) X(matmul_qs_static)               \
  X(quantize_mxfp8) X(quantize_mxfp4) X(quantize_fp8) X(to_bf16) X(decoder_init_model) X(decoder_rmsnorm)       \
  X(decoder_rmsnorm_absmax) X(decoder_softmax_argmax) X(quantize_mxfp6) X(nvfp4_tensor_scales)                  \
  X(nvfp4_tensor_scales_absmax) X(quantize_nvfp4) X(to_bf16_x4) X(matmul_bf16) X(matmul_mxfp6)
L2C_ENTRIES(L2C_ENTRY)

PyObject *initialise(PyObject *, PyObject *args) {
  PyObject *raw = nullptr, *fallback = nullptr;
  if (!PyArg_ParseTuple(args, "OO", &raw, &fallback)) return nullptr;
  Py_INCREF(raw);
  Py_INCREF(fallback);
  Py_XSETREF(g_raw_stream, raw);
  Py_XSETREF(g_fallback, fallback);
  Py_RETURN_NONE;
}

#define L2C_METHOD(NAME) {#NAME, reinterpret_cast<PyCFunction>(py_##NAME), METH_FASTCALL, nullptr},
PyMethodDef methods[] = {L2C_ENTRIES(L2C_METHOD){"initialise", initialise, METH_VARARGS, nullptr},
                         {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "l2c_native", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_l2c_native() {
  g_is_cuda = PyUnicode_InternFromString("is_cuda");
  g_data_ptr = PyUnicode_InternFromString("data_ptr");
  g_cuda_stream = PyUnicode_InternFromString("cuda_stream");
  if (!g_is_cuda || !g_data_ptr || !g_cuda_stream) return nullptr;
  return PyModule_Create(&module);
}
