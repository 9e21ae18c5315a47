// CPython entry points of the library's per-call functions.
//
// A call through ctypes converts 20 to 30 arguments one by one, 3 to 5 us of
// host time where the smallest launches take 5 to 8 us on the GPU.  These
// take the same arguments in the same order, positionally, as Python ints
// (None for a null pointer) and return the function's status; a parameter
// that is a host array of up to PL_MAX_STACKED_MODULES elements (pointers,
// strides, counts of sibling modules) takes a tuple of ints, copied into the
// call's own frame.  The GIL is released around the call.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <limits>
#include <tuple>
#include <type_traits>
#include <utility>

#include "../../include/polylora_hip.h"

namespace {

bool to_int64(PyObject* o, int64_t* out) {
  *out = PyLong_AsLongLong(o);
  return *out != -1 || !PyErr_Occurred();
}

bool to_pointer(PyObject* o, void** out) {
  if (o == Py_None) {
    *out = nullptr;
    return true;
  }
  *out = PyLong_AsVoidPtr(o);
  return *out != nullptr || !PyErr_Occurred();
}

template <typename A>
struct Arg {  // int32_t and int64_t
  static_assert(std::is_integral<A>::value, "integers and pointers only");
  A v;
  bool set(PyObject* o) {
    int64_t w;
    if (!to_int64(o, &w)) return false;
    if (w < std::numeric_limits<A>::min() || w > std::numeric_limits<A>::max()) {
      PyErr_SetString(PyExc_OverflowError, "argument out of range");
      return false;
    }
    v = (A)w;
    return true;
  }
  A get() { return v; }
};

template <typename P>
struct Arg<P*> {  // a pointer, or a host array given as a tuple
  typedef typename std::remove_const<P>::type E;
  void* p;
  int64_t array[PL_MAX_STACKED_MODULES];  // room for 8-byte elements
  bool set(PyObject* o) {
    if (!PyTuple_Check(o)) return to_pointer(o, &p);
    if constexpr (std::is_same<E, int32_t>::value || std::is_same<E, int64_t>::value ||
                  std::is_pointer<E>::value) {
      const Py_ssize_t n = PyTuple_GET_SIZE(o);
      if (n > PL_MAX_STACKED_MODULES) {
        PyErr_SetString(PyExc_ValueError, "too many array elements");
        return false;
      }
      E* e = reinterpret_cast<E*>(array);
      for (Py_ssize_t i = 0; i < n; ++i) {
        PyObject* item = PyTuple_GET_ITEM(o, i);
        if constexpr (std::is_pointer<E>::value) {
          void* q;
          if (!to_pointer(item, &q)) return false;
          e[i] = static_cast<E>(q);
        } else {
          Arg<E> a;
          if (!a.set(item)) return false;
          e[i] = a.get();
        }
      }
      p = array;
      return true;
    } else {
      PyErr_SetString(PyExc_TypeError, "this pointer parameter takes no array");
      return false;
    }
  }
  P* get() { return static_cast<P*>(p); }
};

template <auto Fn>
struct Call;
template <typename... A, int (*Fn)(A...)>
struct Call<Fn> {
  template <size_t... I>
  static PyObject* run(PyObject* const* args, std::index_sequence<I...>) {
    std::tuple<Arg<A>...> a;
    if (!(std::get<I>(a).set(args[I]) && ...)) return nullptr;
    int rc;
    Py_BEGIN_ALLOW_THREADS;
    rc = Fn(std::get<I>(a).get()...);
    Py_END_ALLOW_THREADS;
    return PyLong_FromLong(rc);
  }
  static PyObject* call(PyObject*, PyObject* const* args, Py_ssize_t n) {
    if (n != (Py_ssize_t)sizeof...(A)) {
      PyErr_Format(PyExc_TypeError, "%zd arguments given, %zd taken", n, (Py_ssize_t)sizeof...(A));
      return nullptr;
    }
    return run(args, std::index_sequence_for<A...>());
  }
};

#define PL_CALL(name) \
  {#name, (PyCFunction)(void (*)(void))&Call<&name>::call, METH_FASTCALL, nullptr}

PyMethodDef methods[] = {PL_CALL(pl_lora_apply),
                         PL_CALL(pl_lora_apply_rows),
                         PL_CALL(pl_lora_fused),
                         PL_CALL(pl_lora_fused_stacked),
                         PL_CALL(pl_lora_long_stacked),
                         PL_CALL(pl_lora_decode_stacked),
                         PL_CALL(pl_sgmv_shrink_stacked),
                         PL_CALL(pl_sgmv_expand_stacked),
                         PL_CALL(pl_sgmv_lora_a_ref_parts),
                         PL_CALL(pl_sgmv_lora_b_ref_parts),
                         {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_calls", nullptr, -1, methods,
                      nullptr,               nullptr,  nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__calls(void) { return PyModule_Create(&module); }
