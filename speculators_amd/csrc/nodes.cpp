// Autograd nodes in C++ for the plug-in calls whose kernels take less time than the same nodes cost in Python: the
// attention function and the loss functions behind the reference's registries.  A Python node costs 20 us per direction
// (argument and context objects, the interpreter's lock taken again on the engine's thread); these cost 5.
// 1024 tokens of the 1B attention shape, forward and backward issued: 150 -> 75 us; a loss function 130 -> 75 us.

#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_function.h>

#include "host_common.h"

namespace spx_host {

static const int32_t* i32(const Tensor& t) { return static_cast<const int32_t*>(t.const_data_ptr()); }

Tensor attention_forward(const Tensor& q, const Tensor& k, const Tensor& v, const Mask& m, double scaling,
                         const Tensor& out) {
  const int64_t hq = q.size(1), nq = q.size(2), d = q.size(3), hkv = k.size(1);
  const Tensor lse = at::empty({hq, nq}, q.options().dtype(at::kFloat));
  const bool blocks = m.blo.defined();
  const int64_t n = blocks ? spx_dflash_attn_workspace_bytes(m.T, nq, hq, hkv, d, 0)
                           : spx_ttt_attn_workspace_bytes(nq, hq, hkv, d, 0);
  const Tensor ws = bytes(n, q);
  void* const st = stream_of(q);
  float* const l = lse.mutable_data_ptr<float>();
  if (blocks)
    check(spx_dflash_attn_fwd(q.const_data_ptr(), q.stride(1), k.const_data_ptr(), k.stride(1), v.const_data_ptr(),
                              v.stride(1), i32(m.lo), i32(m.hi), i32(m.blo), i32(m.bhi), m.T, nq, hq, hkv, d, scaling,
                              out.mutable_data_ptr(), l, ws.mutable_data_ptr(), n, st),
          "spx_dflash_attn_fwd");
  else if (m.hi.defined())
    check(spx_span_attn_fwd(q.const_data_ptr(), q.stride(1), k.const_data_ptr(), k.stride(1), v.const_data_ptr(),
                            v.stride(1), i32(m.lo), i32(m.hi), nq, hq, hkv, d, scaling, out.mutable_data_ptr(), l,
                            ws.mutable_data_ptr(), n, st),
          "spx_span_attn_fwd");
  else
    check(spx_ttt_attn_fwd(q.const_data_ptr(), q.stride(1), k.const_data_ptr(), k.stride(1), v.const_data_ptr(),
                           v.stride(1), i32(m.lo), nq, m.step, hq, hkv, d, scaling, out.mutable_data_ptr(), l,
                           ws.mutable_data_ptr(), n, st),
          "spx_ttt_attn_fwd");
  return lse;
}

std::tuple<Tensor, Tensor, Tensor> attention_backward(const Tensor& q, const Tensor& k, const Tensor& v,
                                                      const Tensor& out, const Tensor& dout, const Tensor& lse,
                                                      const Mask& m, double scaling) {
  const int64_t hq = q.size(1), nq = q.size(2), d = q.size(3), hkv = k.size(1);
  const Tensor dq = at::empty_like(q), dk = at::empty_like(k), dv = at::empty_like(v);
  const bool blocks = m.blo.defined();
  const int64_t n = blocks ? spx_dflash_attn_workspace_bytes(m.T, nq, hq, hkv, d, 1)
                           : spx_ttt_attn_workspace_bytes(nq, hq, hkv, d, 1);
  const Tensor ws = bytes(n, q);
  void* const st = stream_of(q);
  const float* const l = lse.const_data_ptr<float>();
  if (blocks)
    check(spx_dflash_attn_bwd(q.const_data_ptr(), q.stride(1), k.const_data_ptr(), k.stride(1), v.const_data_ptr(),
                              v.stride(1), out.const_data_ptr(), dout.const_data_ptr(), l, i32(m.lo), i32(m.hi),
                              i32(m.blo), i32(m.bhi), m.T, nq, hq, hkv, d, scaling, dq.mutable_data_ptr(), dq.stride(1),
                              dk.mutable_data_ptr(), dk.stride(1), dv.mutable_data_ptr(), dv.stride(1),
                              ws.mutable_data_ptr(), n, st),
          "spx_dflash_attn_bwd");
  else if (m.hi.defined())
    check(spx_span_attn_bwd(q.const_data_ptr(), q.stride(1), k.const_data_ptr(), k.stride(1), v.const_data_ptr(),
                            v.stride(1), out.const_data_ptr(), dout.const_data_ptr(), l, i32(m.lo), i32(m.hi), nq, hq,
                            hkv, d, scaling, dq.mutable_data_ptr(), dq.stride(1), dk.mutable_data_ptr(), dk.stride(1),
                            dv.mutable_data_ptr(), dv.stride(1), ws.mutable_data_ptr(), n, st),
          "spx_span_attn_bwd");
  else
    check(spx_ttt_attn_bwd(q.const_data_ptr(), q.stride(1), k.const_data_ptr(), k.stride(1), v.const_data_ptr(),
                           v.stride(1), out.const_data_ptr(), dout.const_data_ptr(), l, i32(m.lo), nq, m.step, hq, hkv,
                           d, scaling, dq.mutable_data_ptr(), dq.stride(1), dk.mutable_data_ptr(), dk.stride(1),
                           dv.mutable_data_ptr(), dv.stride(1), ws.mutable_data_ptr(), n, st),
          "spx_ttt_attn_bwd");
  return {dq, dk, dv};
}

}  // namespace spx_host

namespace {

using namespace spx_host;
using torch::autograd::AutogradContext;
using torch::autograd::Function;
using torch::autograd::variable_list;

// ---------------------------------------------------------------- attention
struct Attention : Function<Attention> {
  static Tensor forward(AutogradContext* ctx, const Tensor& q_, const Tensor& k_, const Tensor& v_, const Tensor& lo,
                        const std::optional<Tensor>& hi_, const std::optional<Tensor>& blo_,
                        const std::optional<Tensor>& bhi_, int64_t T, int64_t step, double scaling) {
    const Mask m{lo, hi_.value_or(Tensor()), blo_.value_or(Tensor()), bhi_.value_or(Tensor()), T, step};
    const Tensor q = q_.contiguous(), k = k_.contiguous(), v = v_.contiguous();
    const Tensor out = at::empty({1, q.size(2), q.size(1), q.size(3)}, q.options());
    const Tensor lse = attention_forward(q, k, v, m, scaling, out);
    ctx->save_for_backward({q, k, v, out, lse, m.lo, m.hi, m.blo, m.bhi});
    ctx->saved_data["T"] = T;
    ctx->saved_data["step"] = step;
    ctx->saved_data["scaling"] = scaling;
    return out;
  }

  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto s = ctx->get_saved_variables();
    const Mask m{s[5], s[6], s[7], s[8], ctx->saved_data["T"].toInt(), ctx->saved_data["step"].toInt()};
    const auto [dq, dk, dv] = attention_backward(s[0], s[1], s[2], s[3], grads[0].to(at::kBFloat16).contiguous(), s[4],
                                                 m, ctx->saved_data["scaling"].toDouble());
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

}  // namespace

PyObject* spx_node_attention(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TORCH_CHECK_TYPE(n == 10, "attention takes 10 arguments");
  const Tensor &q = tensor(args[0]), &k = tensor(args[1]), &v = tensor(args[2]);
  need_hip(q); need_hip(k); need_hip(v); need_hip(tensor(args[3]));
  const int64_t T = PyLong_AsLongLong(args[7]), step = PyLong_AsLongLong(args[8]);
  const double scaling = PyFloat_AsDouble(args[9]);
  if (PyErr_Occurred()) return nullptr;
  const Tensor& lo = tensor(args[3]);
  const auto hi = tensor_or_none(args[4]), block_lo = tensor_or_none(args[5]), block_hi = tensor_or_none(args[6]);
  Unlocked released;
  const Tensor out = Attention::apply(q, k, v, lo, hi, block_lo, block_hi, T, step, scaling);
  released.lock();
  return THPVariable_Wrap(out);
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
  Unlocked released;
  const Tensor out = RowLoss::apply(x, y, op);
  released.lock();
  return THPVariable_Wrap(out);
  END_HANDLE_TH_ERRORS
}

// (ctx.needs_input_grad of a Python node says what requires a gradient, not what this pass was asked for)
PyObject* spx_node_wanted(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TORCH_CHECK_TYPE(n == 1 && THPFunction_Check(args[0]), "wanted takes the context of an autograd function");
  const auto node = reinterpret_cast<THPFunction*>(args[0])->cdata.lock();
  TORCH_CHECK_VALUE(node, "the context belongs to no node of a graph");
  const Py_ssize_t inputs = (Py_ssize_t)node->num_outputs();
  PyObject* const all = PyTuple_New(inputs);
  if (!all) return nullptr;
  for (Py_ssize_t i = 0; i < inputs; ++i) PyTuple_SET_ITEM(all, i, PyBool_FromLong(node->task_should_compute_output(i)));
  return all;
  END_HANDLE_TH_ERRORS
}
