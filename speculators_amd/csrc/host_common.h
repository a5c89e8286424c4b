// What the host code above the entry points shares (nodes.cpp, layer_host.cpp).
#pragma once
#include <Python.h>

#include <utility>

#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/spx.h"
#include "nodes.h"

namespace spx_host {

using at::Tensor;

inline void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

// The error goes through the autograd engine as the Python exception it is.
[[noreturn]] inline void fail(const char* fmt, const char* a, long rc = 0, const char* b = "") {
  PyGILState_STATE g = PyGILState_Ensure();
  PyErr_Format(spx_error_class(), fmt, a, rc, b);
  python_error e;
  e.persist();
  PyGILState_Release(g);
  throw e;
}
inline void check(int rc, const char* name) {
  if (rc != 0) fail("%s failed (%ld): %s", name, rc, spx_last_error());
}
// The interpreter's lock given up, from the construction on until lock() or the end of the scope (by an exception, too).
// No Python object is touched in between; the tensors of the call's arguments stay, its caller holds them.
class Unlocked {
 public:
  Unlocked() : state_(PyEval_SaveThread()) {}
  Unlocked(const Unlocked&) = delete;
  ~Unlocked() { lock(); }
  void lock() {
    if (state_) PyEval_RestoreThread(std::exchange(state_, nullptr));
  }

 private:
  PyThreadState* state_;
};
inline void need_hip(const Tensor& t) {
  if (!t.is_cuda()) fail("%s", "libspx_hip works on HIP device tensors only (got a CPU tensor)");
}
inline Tensor bytes(int64_t n, const Tensor& like) { return at::empty({n}, like.options().dtype(at::kByte)); }

inline const Tensor& tensor(PyObject* o) {
  TORCH_CHECK_TYPE(THPVariable_Check(o), "expected a tensor, got ", Py_TYPE(o)->tp_name);
  return THPVariable_Unpack(o);
}
inline std::optional<Tensor> tensor_or_none(PyObject* o) {
  if (o == Py_None) return std::nullopt;
  return tensor(o);
}

// The mask of an attention call: lo only: TTT (step, T keys per step); lo, hi: one interval per row; blo, bhi too: anchored
// blocks behind T context keys.
struct Mask {
  Tensor lo, hi, blo, bhi;
  int64_t T, step;
};
Tensor attention_forward(const Tensor& q, const Tensor& k, const Tensor& v, const Mask& m, double scaling,
                         const Tensor& out);  // -> row statistics
std::tuple<Tensor, Tensor, Tensor> attention_backward(const Tensor& q, const Tensor& k, const Tensor& v,
                                                      const Tensor& out, const Tensor& dout, const Tensor& lse,
                                                      const Mask& m, double scaling);

}  // namespace spx_host
