// Autograd nodes in C++ for the plug-in calls whose kernels take less time than the same nodes cost in Python: the
// attention function and the loss functions behind the reference's registries.  A Python node costs 20 us per direction
// (argument and context objects, the interpreter's lock taken again on the engine's thread); these cost 5.
// 1024 tokens of the 1B attention shape, forward and backward issued: 150 -> 75 us; a loss function 130 -> 75 us.

#include <Python.h>

#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/spx.h"
#include "nodes.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::Function;
using torch::autograd::variable_list;

void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

// The error goes through the autograd engine as the Python exception it is.
[[noreturn]] void fail(const char* fmt, const char* a, long rc = 0, const char* b = "") {
  PyGILState_STATE g = PyGILState_Ensure();
  PyErr_Format(spx_error_class(), fmt, a, rc, b);
  python_error e;
  e.persist();
  PyGILState_Release(g);
  throw e;
}
void check(int rc, const char* name) {
  if (rc != 0) fail("%s failed (%ld): %s", name, rc, spx_last_error());
}
void need_hip(const Tensor& t) {
  if (!t.is_cuda()) fail("%s", "libspx_hip works on HIP device tensors only (got a CPU tensor)");
}
Tensor bytes(int64_t n, const Tensor& like) { return at::empty({n}, like.options().dtype(at::kByte)); }

// ---------------------------------------------------------------- attention
// lo only: TTT (step, T keys per step); lo, hi: one interval per row; blo, bhi too: anchored blocks behind T context keys
struct Attention : Function<Attention> {
  static Tensor forward(AutogradContext* ctx, const Tensor& q_, const Tensor& k_, const Tensor& v_, const Tensor& lo,
                        const std::optional<Tensor>& hi_, const std::optional<Tensor>& blo_,
                        const std::optional<Tensor>& bhi_, int64_t T, int64_t step, double scaling) {
    const Tensor hi = hi_.value_or(Tensor()), blo = blo_.value_or(Tensor()), bhi = bhi_.value_or(Tensor());
    const Tensor q = q_.contiguous(), k = k_.contiguous(), v = v_.contiguous();
    const int64_t hq = q.size(1), nq = q.size(2), d = q.size(3), hkv = k.size(1);
    const Tensor out = at::empty({1, nq, hq, d}, q.options());
    const Tensor lse = at::empty({hq, nq}, q.options().dtype(at::kFloat));
    const bool blocks = blo.defined(), span = hi.defined();
    const int64_t n = blocks ? spx_dflash_attn_workspace_bytes(T, nq, hq, hkv, d, 0)
                             : spx_ttt_attn_workspace_bytes(nq, hq, hkv, d, 0);
    const Tensor ws = bytes(n, q);
    void* const st = stream_of(q);
    auto i32 = [](const Tensor& t) { return static_cast<const int32_t*>(t.const_data_ptr()); };
    if (blocks)
      check(spx_dflash_attn_fwd(q.const_data_ptr(), q.stride(1), k.const_data_ptr(), k.stride(1), v.const_data_ptr(),
                                v.stride(1), i32(lo), i32(hi), i32(blo), i32(bhi), T, nq, hq, hkv, d, scaling,
                                out.mutable_data_ptr(), lse.mutable_data_ptr<float>(), ws.mutable_data_ptr(), n, st),
            "spx_dflash_attn_fwd");
    else if (span)
      check(spx_span_attn_fwd(q.const_data_ptr(), q.stride(1), k.const_data_ptr(), k.stride(1), v.const_data_ptr(),
                              v.stride(1), i32(lo), i32(hi), nq, hq, hkv, d, scaling, out.mutable_data_ptr(),
                              lse.mutable_data_ptr<float>(), ws.mutable_data_ptr(), n, st),
            "spx_span_attn_fwd");
    else
      check(spx_ttt_attn_fwd(q.const_data_ptr(), q.stride(1), k.const_data_ptr(), k.stride(1), v.const_data_ptr(),
                             v.stride(1), i32(lo), nq, step, hq, hkv, d, scaling, out.mutable_data_ptr(),
                             lse.mutable_data_ptr<float>(), ws.mutable_data_ptr(), n, st),
            "spx_ttt_attn_fwd");
    ctx->save_for_backward({q, k, v, out, lse, lo, hi, blo, bhi});
    ctx->saved_data["T"] = T;
    ctx->saved_data["step"] = step;
    ctx->saved_data["scaling"] = scaling;
    return out;
  }

  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto s = ctx->get_saved_variables();
    const Tensor &q = s[0], &k = s[1], &v = s[2], &out = s[3], &lse = s[4], &lo = s[5], &hi = s[6], &blo = s[7], &bhi = s[8];
    const int64_t T = ctx->saved_data["T"].toInt(), step = ctx->saved_data["step"].toInt();
    const double scaling = ctx->saved_data["scaling"].toDouble();
    const int64_t hq = q.size(1), nq = q.size(2), d = q.size(3), hkv = k.size(1);
    const Tensor dout = grads[0].to(at::kBFloat16).contiguous();
    const Tensor dq = at::empty_like(q), dk = at::empty_like(k), dv = at::empty_like(v);
    const bool blocks = blo.defined(), span = hi.defined();
    const int64_t n = blocks ? spx_dflash_attn_workspace_bytes(T, nq, hq, hkv, d, 1)
                             : spx_ttt_attn_workspace_bytes(nq, hq, hkv, d, 1);
    const Tensor ws = bytes(n, q);
    void* const st = stream_of(q);
    auto i32 = [](const Tensor& t) { return static_cast<const int32_t*>(t.const_data_ptr()); };
    if (blocks)
      check(spx_dflash_attn_bwd(q.const_data_ptr(), q.stride(1), k.const_data_ptr(), k.stride(1), v.const_data_ptr(),
                                v.stride(1), out.const_data_ptr(), dout.const_data_ptr(), lse.const_data_ptr<float>(),
                                i32(lo), i32(hi), i32(blo), i32(bhi), T, nq, hq, hkv, d, scaling, dq.mutable_data_ptr(),
                                dq.stride(1), dk.mutable_data_ptr(), dk.stride(1), dv.mutable_data_ptr(), dv.stride(1),
                                ws.mutable_data_ptr(), n, st),
            "spx_dflash_attn_bwd");
    else if (span)
      check(spx_span_attn_bwd(q.const_data_ptr(), q.stride(1), k.const_data_ptr(), k.stride(1), v.const_data_ptr(),
                              v.stride(1), out.const_data_ptr(), dout.const_data_ptr(), lse.const_data_ptr<float>(),
                              i32(lo), i32(hi), nq, hq, hkv, d, scaling, dq.mutable_data_ptr(), dq.stride(1),
                              dk.mutable_data_ptr(), dk.stride(1), dv.mutable_data_ptr(), dv.stride(1),
                              ws.mutable_data_ptr(), n, st),
            "spx_span_attn_bwd");
    else
      check(spx_ttt_attn_bwd(q.const_data_ptr(), q.stride(1), k.const_data_ptr(), k.stride(1), v.const_data_ptr(),
                             v.stride(1), out.const_data_ptr(), dout.const_data_ptr(), lse.const_data_ptr<float>(),
                             i32(lo), nq, step, hq, hkv, d, scaling, dq.mutable_data_ptr(), dq.stride(1),
                             dk.mutable_data_ptr(), dk.stride(1), dv.mutable_data_ptr(), dv.stride(1),
                             ws.mutable_data_ptr(), n, st),
            "spx_ttt_attn_bwd");
    return {dq, dk, dv, Tensor(), Tensor(), Tensor(), Tensor(), Tensor(), Tensor(), Tensor()};
  }
};

// ---------------------------------------------------------------- row losses
int code_of(const Tensor& t) {
  if (t.scalar_type() == at::kBFloat16) return 0;
  if (t.scalar_type() == at::kFloat) return 1;
  fail("unsupported dtype %s: bf16 and f32 only", c10::toString(t.scalar_type()));
}
// [..., V] -> [rows, V] with unit inner stride (a copy only where the rows are not equally spaced)
Tensor rows_2d(const Tensor& t) {
  return (t.stride(-1) == 1 ? t : t.contiguous()).reshape({-1, t.size(-1)});
}

struct RowLoss : Function<RowLoss> {
  static Tensor forward(AutogradContext* ctx, const Tensor& logits, const Tensor& targets, int64_t op) {
    const Tensor x = rows_2d(logits), y = rows_2d(targets.to(logits.scalar_type()));
    const int64_t rows = x.size(0), vocab = x.size(1);
    const Tensor stats = at::empty({4, rows}, x.options().dtype(at::kFloat));
    const Tensor arg = at::empty({2, rows}, x.options().dtype(at::kInt));
    float* const s = stats.mutable_data_ptr<float>();
    int32_t* const a = arg.mutable_data_ptr<int32_t>();
    check(spx_fused_vocab_loss_fwd(op, x.const_data_ptr(), x.stride(0), y.const_data_ptr(), y.stride(0), rows, vocab,
                                   code_of(x), s, s + rows, s + 2 * rows, s + 3 * rows, a, a + rows, 0, stream_of(x)),
          "spx_fused_vocab_loss_fwd");
    ctx->save_for_backward({x, y, stats, arg});
    ctx->saved_data["op"] = op;
    return stats.select(0, 0).view(logits.sizes().slice(0, logits.dim() - 1));
  }

  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    const Tensor &x = saved[0], &y = saved[1], &stats = saved[2], &arg = saved[3];
    const int64_t rows = x.size(0), vocab = x.size(1);
    const Tensor g = grads[0].reshape({-1}).to(at::kFloat).contiguous();
    const Tensor grad = at::empty({rows, vocab}, x.options());
    const float* const s = stats.const_data_ptr<float>();
    check(spx_fused_vocab_loss_bwd(ctx->saved_data["op"].toInt(), x.const_data_ptr(), x.stride(0), y.const_data_ptr(),
                                   y.stride(0), rows, vocab, code_of(x), s + rows, s + 2 * rows, s + 3 * rows,
                                   arg.const_data_ptr<int32_t>() + rows, g.const_data_ptr<float>(), nullptr,
                                   grad.mutable_data_ptr(), vocab, stream_of(x)),
          "spx_fused_vocab_loss_bwd");
    auto shape = grads[0].sizes().vec();
    shape.push_back(vocab);
    return {grad.view(shape), Tensor(), Tensor()};
  }
};

const Tensor& tensor(PyObject* o) {
  TORCH_CHECK_TYPE(THPVariable_Check(o), "expected a tensor, got ", Py_TYPE(o)->tp_name);
  return THPVariable_Unpack(o);
}
std::optional<Tensor> tensor_or_none(PyObject* o) {
  if (o == Py_None) return std::nullopt;
  return tensor(o);
}

}  // namespace

PyObject* spx_node_attention(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TORCH_CHECK_TYPE(n == 10, "attention takes 10 arguments");
  const Tensor &q = tensor(args[0]), &k = tensor(args[1]), &v = tensor(args[2]);
  need_hip(q); need_hip(k); need_hip(v); need_hip(tensor(args[3]));
  const int64_t T = PyLong_AsLongLong(args[7]), step = PyLong_AsLongLong(args[8]);
  const double scaling = PyFloat_AsDouble(args[9]);
  if (PyErr_Occurred()) return nullptr;
  return THPVariable_Wrap(Attention::apply(q, k, v, tensor(args[3]), tensor_or_none(args[4]),
                                           tensor_or_none(args[5]), tensor_or_none(args[6]), T, step, scaling));
  END_HANDLE_TH_ERRORS
}

PyObject* spx_node_row_loss(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TORCH_CHECK_TYPE(n == 3, "row_loss takes 3 arguments");
  const int64_t op = PyLong_AsLongLong(args[0]);
  if (op == -1 && PyErr_Occurred()) return nullptr;
  const Tensor &x = tensor(args[1]), &y = tensor(args[2]);
  TORCH_CHECK_VALUE(x.sizes() == y.sizes(), "logits ", x.sizes(), " and targets ", y.sizes(), " differ");
  need_hip(x); need_hip(y);
  return THPVariable_Wrap(RowLoss::apply(x, y, op));
  END_HANDLE_TH_ERRORS
}
