// CPython extension deers_amd._calls: the entry points of include/deers_rocm.h that a training step or
// a generated token consists of, as built-in functions.
//
// A generated token is about 110 such calls, each a few microseconds of GPU time, and ctypes spends
// more than a microsecond of a call on making and unpacking its argument objects.  Here the arguments are
// converted by the C type that each parameter has, without intermediate objects: the host part of a
// token (32 sequences, 12 blocks) 433 -> 378 us, of a forward and backward of attention 11-13 -> 9 us.  The functions raise the binding's error class on a
// non-zero return code and release the interpreter lock during the call, as ctypes does.
//
//   pointers    None, an int or a ctypes.c_void_p; for anything else the binding's `address` says which
//               address it stands for, or refuses it.  An object's own storage is host memory, which a
//               kernel must not be given.
//   dimensions  None or a sequence of what int() takes, copied for the duration of the call
//   sizes       a sequence of ints
//   tables      a sequence of pointers
//   dtoh's destination, the one host buffer: an object with a writable buffer that holds the bytes
//
// The library is the one the binding has loaded: bind(path, c_void_p, error class, address) looks the
// functions up in it, so that the path can be chosen at run time.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <dlfcn.h>

#include <array>
#include <tuple>
#include <utility>
#include <vector>

#include "../../include/deers_rocm.h"

namespace {

PyTypeObject* g_void_p = nullptr;  // ctypes.c_void_p
PyObject* g_error = nullptr;       // the exception class for a non-zero return code
PyObject* g_address = nullptr;     // address(object) -> int
decltype(&deers_rocm_last_error) g_last_error = nullptr;

bool to_int64(PyObject* o, int64_t* out) {
  *out = PyLong_AsLongLong(o);
  return *out != -1 || !PyErr_Occurred();
}
// As int(o), which strides have always been passed through.
bool to_dimension(PyObject* o, int64_t* out) {
  if (PyLong_Check(o)) return to_int64(o, out);
  PyObject* i = PyNumber_Long(o);
  const bool ok = i && to_int64(i, out);
  Py_XDECREF(i);
  return ok;
}
bool to_address(PyObject* o, void** out) {
  if (o == Py_None) {
    *out = nullptr;
    return true;
  }
  if (PyLong_Check(o)) {
    *out = PyLong_AsVoidPtr(o);
    return *out || !PyErr_Occurred();
  }
  if (Py_IS_TYPE(o, g_void_p)) {
    Py_buffer view;  // of the eight bytes that hold the address
    if (PyObject_GetBuffer(o, &view, PyBUF_SIMPLE) != 0) return false;
    *out = *(void**)view.buf;
    PyBuffer_Release(&view);
    return true;
  }
  PyObject* address = PyObject_CallOneArg(g_address, o);
  if (!address) return false;
  *out = PyLong_AsVoidPtr(address);
  Py_DECREF(address);
  return *out || !PyErr_Occurred();
}

// One converter per kind of parameter: from() fills it, get() is what the C function takes.
struct Int {
  int64_t v = 0;
  bool from(PyObject* o) {
    if (!to_int64(o, &v)) return false;
    if (v < INT32_MIN || v > INT32_MAX) {
      PyErr_SetString(PyExc_OverflowError, "value does not fit an int");
      return false;
    }
    return true;
  }
  int get() { return (int)v; }
};
struct Int64 {
  int64_t v = 0;
  bool from(PyObject* o) { return to_int64(o, &v); }
  int64_t get() { return v; }
};
struct Size {
  int64_t v = 0;
  bool from(PyObject* o) { return to_int64(o, &v); }
  size_t get() { return (size_t)v; }
};
struct Double {
  double v = 0;
  bool from(PyObject* o) {
    v = PyFloat_AsDouble(o);
    return v != -1.0 || !PyErr_Occurred();
  }
  double get() { return v; }
};
struct Float : Double {
  float get() { return (float)v; }
};
template <class T>
struct Ptr {
  void* v = nullptr;
  bool from(PyObject* o) { return to_address(o, &v); }
  T* get() { return static_cast<T*>(v); }
};
// Host memory to be written, held until the call is over.
struct HostOut {
  Py_buffer view{};
  bool from(PyObject* o) {
    if (PyObject_TypeCheck(o, g_void_p)) {  // its buffer is the address it holds
      PyErr_SetString(PyExc_TypeError, "the destination is an object with a writable buffer, not an address");
      return false;
    }
    return PyObject_GetBuffer(o, &view, PyBUF_WRITABLE) == 0;
  }
  void* get() { return view.buf; }
  ~HostOut() { PyBuffer_Release(&view); }
};

// A sequence as a tuple or list, checked for its length (N = 0: any).
PyObject* sequence(PyObject* o, size_t n) {
  PyObject* s = PySequence_Fast(o, "a sequence is needed");
  if (s && n && (size_t)PySequence_Fast_GET_SIZE(s) != n) {
    PyErr_Format(PyExc_ValueError, "%zu dimensions are needed, not %zd", n, PySequence_Fast_GET_SIZE(s));
    Py_CLEAR(s);
  }
  return s;
}
template <class V, bool (*CONVERT)(PyObject*, V*), size_t N>
struct Items {
  std::array<V, N ? N : 128> few;
  std::vector<V> many;
  V* v = nullptr;
  bool from(PyObject* o) {
    PyObject* s = sequence(o, N);
    if (!s) return false;
    const Py_ssize_t n = PySequence_Fast_GET_SIZE(s);
    v = few.data();
    if ((size_t)n > few.size()) {
      many.resize((size_t)n);
      v = many.data();
    }
    bool ok = true;
    for (Py_ssize_t i = 0; ok && i < n; ++i) {
      if (i >= PySequence_Fast_GET_SIZE(s)) {  // a conversion may run code that changes a list
        PyErr_SetString(PyExc_RuntimeError, "a list changed its size while it was read");
        ok = false;
        break;
      }
      PyObject* item = PySequence_Fast_GET_ITEM(s, i);
      Py_INCREF(item);
      ok = CONVERT(item, v + i);
      Py_DECREF(item);
    }
    Py_DECREF(s);
    return ok;
  }
};
template <size_t N>
struct Dims : Items<int64_t, to_dimension, N> {  // None: null
  bool from(PyObject* o) { return o == Py_None || Items<int64_t, to_dimension, N>::from(o); }
  const int64_t* get() { return this->v; }
};
struct Sizes : Items<int64_t, to_int64, 0> {
  const int64_t* get() { return v; }
};
template <class T>
struct Table : Items<void*, to_address, 0> {
  T get() { return (T)this->v; }
};

using CP = Ptr<const void>;
using MP = Ptr<void>;
using FP = Ptr<float>;
using CFP = Ptr<const float>;
using IP = Ptr<const int64_t>;  // index vectors in device memory
using I64 = Int64;

template <class... Kinds>
bool fits(std::tuple<Kinds...>&) {
  return true;
}
bool fits(std::tuple<HostOut, CP, Size>& k) {
  if (std::get<0>(k).view.len >= 0 && (size_t)std::get<0>(k).view.len >= std::get<2>(k).get()) return true;
  PyErr_Format(PyExc_ValueError, "%zu bytes do not fit a buffer of %zd", std::get<2>(k).get(), std::get<0>(k).view.len);
  return false;
}

template <class Kinds, class Fn, size_t... I>
PyObject* call(Fn fn, PyObject* const* args, Py_ssize_t n, std::index_sequence<I...>) {
  if (n != (Py_ssize_t)sizeof...(I)) {
    PyErr_Format(PyExc_TypeError, "%zu arguments are needed, not %zd", sizeof...(I), n);
    return nullptr;
  }
  if (!fn) return PyErr_Format(PyExc_RuntimeError, "bind() comes first");
  Kinds k;
  if (!((std::get<I>(k).from(args[I]) && ...) && fits(k))) return nullptr;
  PyThreadState* state = PyEval_SaveThread();
  const int rc = fn(std::get<I>(k).get()...);
  PyEval_RestoreThread(state);
  if (rc != DEERS_ROCM_OK) {
    PyErr_Format(g_error, "deers_rocm error %d: %s", rc, g_last_error());
    return nullptr;
  }
  Py_RETURN_NONE;
}

// X(name, parameter kinds ...)
#define CALLS(X)                                                                                                    \
  X(attn_fwd, Int, CP, Dims<4>, CP, Dims<4>, CP, Dims<4>, MP, Dims<4>, FP, I64, I64, I64, I64, Float)               \
  X(attn_bwd, Int, CP, Dims<4>, CP, Dims<4>, CP, Dims<4>, CP, Dims<4>, CFP, CP, Dims<4>, MP, Dims<4>, MP, Dims<4>,  \
    MP, Dims<4>, I64, I64, I64, I64, Float)                                                                         \
  X(attn_decode, Int, CP, CP, CP, Dims<3>, MP, I64, I64, I64, I64, Float)                                           \
  X(attn_decode_append, Int, CP, CP, CP, Dims<2>, CP, CP, MP, MP, Dims<3>, MP, I64, I64, I64, I64, I64, Float)      \
  X(fill, Int, MP, Size, Float)                                                                                     \
  X(index_select, Int, CP, IP, MP, I64, I64, I64)                                                                   \
  X(index_add, Int, CP, IP, MP, I64, I64, I64)                                                                      \
  X(rms_norm_fwd, Int, CP, MP, I64, I64, Double)                                                                    \
  X(rms_norm_bwd, Int, CP, CP, MP, I64, I64, Double)                                                                \
  X(rms_norm_bwd_add, Int, CP, CP, CP, MP, I64, I64, Double)                                                        \
  X(relu_sq_fwd, Int, CP, MP, I64)                                                                                  \
  X(relu_sq_bwd, Int, CP, CP, MP, I64)                                                                              \
  X(argmax_rows, Int, CP, Ptr<int64_t>, I64, I64)                                                                   \
  X(cross_entropy_fwd, Int, CP, IP, FP, FP, I64, I64)                                                               \
  X(cross_entropy_fwd_grad, Int, CP, IP, FP, FP, MP, I64, I64)                                                      \
  X(cross_entropy_bwd, Int, CP, IP, CFP, CFP, MP, I64, I64)                                                         \
  X(scale_by_scalar, Int, MP, I64, CFP)                                                                             \
  X(adamw_step_multi, Int, Int, Table<void* const*>, Table<const void* const*>, Table<void* const*>,                \
    Table<void* const*>, Sizes, Double, Double, Double, Double, Double, I64, Double)                              \
  X(sum_squares_multi, Int, Int, Table<const void* const*>, Sizes, FP, Int)                                       \
  X(copy_view, Int, CP, Dims<0>, MP, Dims<0>, Dims<0>, Int)                                                         \
  X(matmul, Int, CP, I64, I64, I64, CP, I64, I64, I64, MP, I64, I64, I64, I64)                                      \
  X(matmul_acc, Int, CP, I64, I64, I64, CP, I64, I64, I64, MP, I64, I64, I64, I64)                                  \
  X(matmul_add, Int, CP, I64, I64, I64, CP, I64, I64, I64, CP, MP, I64, I64, I64, I64)                              \
  X(decode_linear, Int, Int, Float, CP, I64, CP, I64, MP, Int, I64, I64, I64)                                       \
  X(decode_linear_hint, CP, I64, I64)                                                                               \
  X(decode_qkv, Int, CP, CP, CP, Dims<2>, CP, CP, MP, MP, MP, Dims<3>, I64, I64, I64, I64, I64)                     \
  X(rope_fwd, Int, CP, Dims<4>, CP, CP, MP, Dims<4>, I64, I64, I64, I64)                                            \
  X(rope_bwd, Int, CP, Dims<4>, CP, CP, MP, I64, I64, I64, I64)                                                     \
  X(dtoh, HostOut, CP, Size)

#define DEFINE(name, ...)                                                                       \
  decltype(&deers_rocm_##name) p_##name = nullptr;                                              \
  PyObject* call_##name(PyObject*, PyObject* const* args, Py_ssize_t n) {                       \
    using Kinds = std::tuple<__VA_ARGS__>;                                                      \
    return call<Kinds>(p_##name, args, n, std::make_index_sequence<std::tuple_size_v<Kinds>>{}); \
  }
CALLS(DEFINE)
#undef DEFINE

PyObject* bind(PyObject*, PyObject* args) {
  const char* path;
  PyObject *void_p, *error, *address;
  if (!PyArg_ParseTuple(args, "sOOO", &path, &void_p, &error, &address)) return nullptr;
  if (!PyType_Check(void_p)) return PyErr_Format(PyExc_TypeError, "c_void_p is needed");
  void* lib = dlopen(path, RTLD_NOW | RTLD_LOCAL);
  if (!lib) return PyErr_Format(PyExc_OSError, "%s", dlerror());
  bool ok = (g_last_error = (decltype(g_last_error))dlsym(lib, "deers_rocm_last_error"));
#define LOOK_UP(name, ...) ok = ok && (p_##name = (decltype(p_##name))dlsym(lib, "deers_rocm_" #name));
  CALLS(LOOK_UP)
#undef LOOK_UP
  if (!ok) return PyErr_Format(PyExc_OSError, "%s: %s", path, dlerror());
  Py_INCREF(void_p);
  Py_XSETREF(g_void_p, (PyTypeObject*)void_p);
  Py_INCREF(error);
  Py_XSETREF(g_error, error);
  Py_INCREF(address);
  Py_XSETREF(g_address, address);
  Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"bind", bind, METH_VARARGS, "bind(path, c_void_p, error, address): look the functions up in the library at `path`"},
#define METHOD(name, ...) {#name, (PyCFunction)(void (*)(void))call_##name, METH_FASTCALL, "deers_rocm_" #name},
    CALLS(METHOD)
#undef METHOD
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_calls", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__calls(void) { return PyModule_Create(&module_def); }
