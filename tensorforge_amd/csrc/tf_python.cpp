// CPython binding of the C ABI for the kernels' Python entry points.
//
// A call through ctypes converts every argument by its declared type: 2.6 us
// for the 11 arguments of a projection and 4.9 us for the 25 of an attention
// call, as much host time as the launch itself.  Here each entry point is a
// vectorcall function whose conversions come from its C prototype at compile
// time.  Pointers are Python integers (addresses) or None; the GIL is
// released around the call, which enqueues work and does not wait.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <cstdint>
#include <tuple>
#include <utility>

#include "../../include/tensorforge_amd.h"

namespace {

// One Python argument as a value of the prototype's type; false with an
// exception set where it is not one.
template <typename T>
bool convert(PyObject *object, T *&out) {
  if (object == Py_None) {
    out = nullptr;
    return true;
  }
  out = static_cast<T *>(PyLong_AsVoidPtr(object));
  return out != nullptr || !PyErr_Occurred();
}

bool convert(PyObject *object, int64_t &out) {
  out = PyLong_AsLongLong(object);
  return out != -1 || !PyErr_Occurred();
}

bool convert(PyObject *object, int32_t &out) {
  int64_t wide = 0;
  if (!convert(object, wide)) return false;
  out = static_cast<int32_t>(wide);
  if (out == wide) return true;
  PyErr_SetString(PyExc_OverflowError, "value does not fit 32 bits");
  return false;
}

bool convert(PyObject *object, float &out) {
  const double wide = PyFloat_AsDouble(object);
  out = static_cast<float>(wide);
  return wide != -1.0 || !PyErr_Occurred();
}

template <auto F>
struct Entry;

template <typename... Args, int32_t (*F)(Args...)>
struct Entry<F> {
  static PyObject *call(PyObject *, PyObject *const *args, Py_ssize_t count) {
    if (count != static_cast<Py_ssize_t>(sizeof...(Args))) {
      PyErr_Format(PyExc_TypeError, "expected %zd arguments, got %zd",
                   static_cast<Py_ssize_t>(sizeof...(Args)), count);
      return nullptr;
    }
    return run(args, std::index_sequence_for<Args...>{});
  }

 private:
  template <std::size_t... I>
  static PyObject *run(PyObject *const *args, std::index_sequence<I...>) {
    std::tuple<Args...> values;
    if (!(convert(args[I], std::get<I>(values)) && ...)) return nullptr;
    int32_t status;
    Py_BEGIN_ALLOW_THREADS
    status = F(std::get<I>(values)...);
    Py_END_ALLOW_THREADS
    return PyLong_FromLong(status);
  }
};

#define TF_ENTRY(name) \
  {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&Entry<&name>::call)), METH_FASTCALL, nullptr}

PyMethodDef methods[] = {
    TF_ENTRY(tf_paged_gqa_decode),
    TF_ENTRY(tf_paged_gqa_decode_rope_append),
    TF_ENTRY(tf_paged_gqa_decode_variant),
    TF_ENTRY(tf_paged_kv_write_token),
    TF_ENTRY(tf_paged_kv_write_slots),
    TF_ENTRY(tf_paged_kv_write_range),
    TF_ENTRY(tf_rope_kv_append),
    TF_ENTRY(tf_rms_norm),
    TF_ENTRY(tf_embedding_rms_norm),
    TF_ENTRY(tf_residual_rms_norm),
    TF_ENTRY(tf_residual_rms_norm_partials),
    TF_ENTRY(tf_swiglu),
    TF_ENTRY(tf_swiglu_rows),
    TF_ENTRY(tf_argmax_rows),
    TF_ENTRY(tf_linear_rows),
    TF_ENTRY(tf_linear_partials),
    TF_ENTRY(tf_linear_partials_sum),
    TF_ENTRY(tf_linear_stream),
    TF_ENTRY(tf_linear_swiglu),
    TF_ENTRY(tf_linear_kstream),
    TF_ENTRY(tf_linear_kstream_norm),
    TF_ENTRY(tf_linear_kstream_residual),
    TF_ENTRY(tf_linear_kswiglu),
    TF_ENTRY(tf_linear_kswiglu_norm),
    TF_ENTRY(tf_prefill_attention),
    TF_ENTRY(tf_prefill_linear),
    TF_ENTRY(tf_prefill_linear_splits),
    TF_ENTRY(tf_prefill_layer),
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_tf_launch", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__tf_launch() { return PyModule_Create(&module); }
