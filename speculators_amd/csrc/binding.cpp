// Python binding of the C entry points (include/spx.h): module speculators_amd._spx_native.
//
// Every entry point becomes a function that takes its arguments positionally -- integers, floats, None (a null
// pointer), or a HIP tensor where the C function takes a pointer -- converts them without an intermediate object, calls
// the function and raises SpxError when its status is not zero.  A call costs what the launch costs: 6.9 us through
// ctypes (argument objects, the foreign call, the status check in Python), 3 us here; a training step of a small draft
// makes a hundred of them.  Entry points that launch are called without the interpreter's lock: a launch that waits for
// room in the queue, or a file that is read, does not hold up the program's other threads (the batch producer's).

#include <Python.h>

#include <torch/csrc/autograd/python_variable.h>

#include <tuple>
#include <type_traits>
#include <utility>

#include "../../include/spx.h"
#include "nodes.h"

namespace {

PyObject* g_error = nullptr;  // SpxError

template <typename T>
bool convert(PyObject* o, T& out) {
  if constexpr (std::is_pointer_v<T>) {
    if (o == Py_None) {
      out = nullptr;
    } else if (PyLong_Check(o)) {
      out = reinterpret_cast<T>(PyLong_AsVoidPtr(o));
      return out != nullptr || !PyErr_Occurred();
    } else if (THPVariable_Check(o)) {
      const at::Tensor& t = THPVariable_Unpack(o);
      if (!t.is_cuda()) {
        PyErr_SetString(g_error, "libspx_hip works on HIP device tensors only (got a CPU tensor)");
        return false;
      }
      out = reinterpret_cast<T>(const_cast<void*>(t.const_data_ptr()));
    } else {
      PyErr_Format(PyExc_TypeError, "expected a tensor, an address or None, got %s", Py_TYPE(o)->tp_name);
      return false;
    }
    return true;
  } else if constexpr (std::is_floating_point_v<T>) {
    out = static_cast<T>(PyFloat_AsDouble(o));
    return !(out == T(-1) && PyErr_Occurred());
  } else {
    const long long v = PyLong_AsLongLong(o);
    out = static_cast<T>(v);
    return !(v == -1 && PyErr_Occurred());
  }
}

template <bool kStatus, auto kFn, typename R, typename... A>
PyObject* call_with(const char* name, PyObject* const* args, Py_ssize_t n, R (*)(A...)) {
  constexpr Py_ssize_t kArgs = sizeof...(A);
  if (n != kArgs) {
    PyErr_Format(PyExc_TypeError, "%s takes %zd arguments (%zd given)", name, kArgs, n);
    return nullptr;
  }
  std::tuple<std::decay_t<A>...> v;
  const bool ok = [&]<size_t... I>(std::index_sequence<I...>) {
    return (convert(args[I], std::get<I>(v)) && ...);
  }(std::make_index_sequence<sizeof...(A)>{});
  if (!ok) return nullptr;
  R r;
  if constexpr (kStatus) {
    Py_BEGIN_ALLOW_THREADS
    r = std::apply(kFn, v);
    Py_END_ALLOW_THREADS
  } else {
    r = std::apply(kFn, v);
  }
  if constexpr (std::is_same_v<R, const char*>) return PyUnicode_FromString(r);
  else if constexpr (std::is_floating_point_v<R>) return PyFloat_FromDouble(r);
  else return PyLong_FromLongLong(r);
}

// kStatus: the result is a status, not a value
template <bool kStatus, auto kFn>
PyObject* entry(const char* name, PyObject* const* args, Py_ssize_t n) {
  PyObject* r = call_with<kStatus, kFn>(name, args, n, kFn);
  if constexpr (kStatus) {
    if (!r) return nullptr;
    const long rc = PyLong_AsLong(r);
    Py_DECREF(r);
    if (rc != 0) {
      PyErr_Format(g_error, "%s failed (%ld): %s", name, rc, spx_last_error());
      return nullptr;
    }
    Py_RETURN_NONE;
  }
  return r;
}

#define SPX_STATUS(fn)                                                                       \
  static PyObject* py_##fn(PyObject*, PyObject* const* args, Py_ssize_t n) {                \
    return entry<true, &fn>(#fn, args, n);                                                  \
  }
#define SPX_VALUE(fn)                                                                        \
  static PyObject* py_##fn(PyObject*, PyObject* const* args, Py_ssize_t n) {                \
    return entry<false, &fn>(#fn, args, n);                                                 \
  }
#include "binding_list.h"
#undef SPX_STATUS
#undef SPX_VALUE

PyObject* set_error(PyObject*, PyObject* cls) {
  Py_INCREF(cls);
  Py_XDECREF(g_error);
  g_error = cls;
  Py_RETURN_NONE;
}

#define SPX_ROW(fn) {#fn, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&py_##fn)), METH_FASTCALL, nullptr},
#define SPX_HOST(name, fn) \
  {name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&fn)), METH_FASTCALL, nullptr},
#define SPX_STATUS(fn) SPX_ROW(fn)
#define SPX_VALUE(fn) SPX_ROW(fn)
PyMethodDef g_methods[] = {
#include "binding_list.h"
    SPX_HOST("attention", spx_node_attention)
    SPX_HOST("row_loss", spx_node_row_loss)
    SPX_HOST("wanted", spx_node_wanted)
    SPX_HOST("product", spx_layer_product)
    SPX_HOST("tail_forward", spx_layer_tail_forward)
    SPX_HOST("tail_backward", spx_layer_tail_backward)
    SPX_HOST("ttt_forward", spx_layer_ttt_forward)
    SPX_HOST("ttt_backward", spx_layer_ttt_backward)
    SPX_HOST("normed_forward", spx_layer_normed_forward)
    SPX_HOST("normed_backward", spx_layer_normed_backward)
    SPX_HOST("product_tn", spx_layer_product_tn)
    SPX_HOST("products_tn", spx_layer_products_tn)
    SPX_HOST("loss_step", spx_layer_loss_step)
    SPX_HOST("loss_terms", spx_layer_loss_terms)
    SPX_HOST("loss_steps_begin", spx_layer_loss_steps_begin)
    SPX_HOST("loss_steps_pass", spx_layer_loss_steps_pass)
    SPX_HOST("loss_steps_end", spx_layer_loss_steps_end)
    SPX_HOST("cat_bf16", spx_layer_cat_bf16)
    SPX_HOST("gain_sums", spx_layer_gain_sums)
    {"set_error", set_error, METH_O, "the exception class raised for a failed call"},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_spx_native", nullptr, -1, g_methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyObject* spx_error_class() { return g_error; }

PyMODINIT_FUNC PyInit__spx_native() {
  g_error = PyExc_RuntimeError;
  Py_INCREF(g_error);
  return PyModule_Create(&g_module);
}
