// The launches of a decoder layer in sequence: what the Python nodes of layer.py run between their bookkeeping.  A launch
// out of Python costs 10 us with the tensor it writes, its strides and addresses (2 us for the tensor, 3 to 5 for the
// call); from here it costs the launch, 3 to 4 us.  Up to a thousand tokens a draft's step was bound by that: 512 tokens of
// the 1B shape, three TTT steps: 2.50 ms -> 2.36 a pass; three layers of anchored blocks over 1777: 3.76 -> 3.61.

#include <algorithm>
#include <vector>

#include "host_common.h"

namespace {

using namespace spx_host;

struct Args {
  PyObject* const* at;
  const char* name;
  Args(const char* fn, PyObject* const* args, Py_ssize_t n, Py_ssize_t want) : at(args), name(fn) {
    TORCH_CHECK_TYPE(n == want, fn, " takes ", want, " arguments (", n, " given)");
  }
  const Tensor& tensor() {
    const Tensor& t = spx_host::tensor(*at++);
    need_hip(t);
    return t;
  }
  Tensor maybe() {
    PyObject* const o = *at++;
    if (o == Py_None) return Tensor();
    const Tensor& t = spx_host::tensor(o);
    need_hip(t);
    return t;
  }
  int64_t integer() {
    const long long v = PyLong_AsLongLong(*at++);
    if (v == -1 && PyErr_Occurred()) throw python_error();
    return v;
  }
  double number() {
    const double v = PyFloat_AsDouble(*at++);
    if (v == -1.0 && PyErr_Occurred()) throw python_error();
    return v;
  }
};

PyObject* wrapped(Unlocked& released, const Tensor& t) {
  released.lock();
  return THPVariable_Wrap(t);
}
PyObject* tuple_of(Unlocked& released, std::initializer_list<Tensor> ts) {
  released.lock();
  PyObject* const out = PyTuple_New(ts.size());
  Py_ssize_t i = 0;
  for (const Tensor& t : ts) PyTuple_SET_ITEM(out, i++, THPVariable_Wrap(t));
  return out;
}

const uint16_t* in(const Tensor& t) { return static_cast<const uint16_t*>(t.const_data_ptr()); }
uint16_t* to(const Tensor& t) { return static_cast<uint16_t*>(t.mutable_data_ptr()); }
float* floats(const Tensor& t) { return t.defined() ? t.mutable_data_ptr<float>() : nullptr; }
Tensor rows_or_new(const Tensor& slot, int64_t rows, int64_t cols, const Tensor& like) {
  return slot.defined() ? slot : at::empty({rows, cols}, like.options().dtype(at::kBFloat16));
}
// [.., H] -> [rows, H] with unit inner stride, bf16
Tensor grad_rows(const Tensor& g) {
  const Tensor x = g.reshape({-1, g.size(-1)}).to(at::kBFloat16);
  return x.stride(1) == 1 ? x : x.contiguous();
}

// A product's result: stored, or (count > 1) as that many partial results in the thread's workspace, which the next launch
// reads.
struct Parted {
  Tensor stored;
  const float* at = nullptr;
  int32_t count = 1;
};

// sum = a + b, y = its norm
void add_norm(const Tensor& a, const Parted& b, const Tensor& sum, const Tensor& gain, const Tensor& y, float* rstd, double eps,
              void* st) {
  const int64_t rows = a.size(0), h = a.size(1);
  if (b.count > 1)
    check(spx_add_rmsnorm_fwd_parts(in(a), a.stride(0), b.at, b.count, to(sum), h, in(gain), to(y), h, rstd, rows, h, eps, st),
          "spx_add_rmsnorm_fwd_parts");
  else
    check(spx_add_rmsnorm_fwd(in(a), a.stride(0), in(b.stored), h, to(sum), h, in(gain), to(y), h, rstd, rows, h, eps, st),
          "spx_add_rmsnorm_fwd");
}

// The backward of a norm over x [rows, h], dres (may be undefined) added to dx; the partial sums of the gain's gradient go
// to scratch (undefined: the gain does not train).
void norm_backward(const Tensor& x, const Tensor& gain, const Tensor& dy, const Tensor& dres, const float* rstd,
                   const Tensor& dx, const Tensor& scratch, int64_t accumulate, void* st) {
  const int64_t rows = x.size(0), h = x.size(1), ld_dres = dres.defined() ? dres.stride(0) : 0;
  const uint16_t* const res = dres.defined() ? in(dres) : nullptr;
  if (scratch.defined())
    check(spx_rmsnorm_bwd_partial(in(x), h, in(gain), in(dy), dy.stride(0), res, ld_dres, rstd, to(dx), h, floats(scratch),
                                  accumulate, rows, h, st),
          "spx_rmsnorm_bwd_partial");
  else
    check(spx_add_rmsnorm_bwd(in(x), h, in(gain), in(dy), dy.stride(0), res, ld_dres, rstd, to(dx), h, nullptr, nullptr, rows,
                              h, st),
          "spx_add_rmsnorm_bwd");
}

void norm_backward(const Tensor& x, const Tensor& gain, const Parted& dy, const Tensor& dres, const float* rstd,
                   const Tensor& dx, const Tensor& scratch, int64_t accumulate, void* st) {
  if (dy.count == 1) return norm_backward(x, gain, dy.stored, dres, rstd, dx, scratch, accumulate, st);
  const int64_t rows = x.size(0), h = x.size(1);
  check(spx_rmsnorm_bwd_parts(in(x), h, in(gain), dy.at, dy.count, dres.defined() ? in(dres) : nullptr,
                              dres.defined() ? dres.stride(0) : 0, rstd, to(dx), h, floats(scratch), accumulate, rows, h, st),
        "spx_rmsnorm_bwd_parts");
}

// How gemm.py routed a product (``Route`` there)
enum { kAutoNT, kAutoNN, kNT, kTail, kLinear, kMatmul, kPairNN, kGatedNT };
struct Products {
  int64_t parts;
  Tensor ws;  // fp32 partials of products cut along the contraction
  Tensor operator()(int64_t route, const Tensor& a, const Tensor& b, const Tensor& m_live = Tensor()) const {
    if (route == kLinear) return at::linear(a, b);
    if (route == kMatmul) return at::matmul(a, b);
    const int64_t m = a.size(0), k = a.size(1), n = route == kAutoNN ? b.size(1) : b.size(0);
    TORCH_CHECK_VALUE(b.size(route == kAutoNN ? 0 : 1) == k, "shape mismatch: a ", a.sizes(), " b ", b.sizes());
    const Tensor out = at::empty({m, n}, a.options());
    void* const st = stream_of(a);
    void* const w = ws.defined() ? ws.mutable_data_ptr() : nullptr;
    const int64_t wb = ws.defined() ? ws.nbytes() : 0;
    if (route == kNT)
      check(spx_gemm_bf16_nt(in(a), a.stride(0), in(b), b.stride(0), to(out), n, m, n, k, st), "spx_gemm_bf16_nt");
    else if (route == kTail)
      check(spx_gemm_bf16_nt_tail(in(a), a.stride(0), in(b), b.stride(0), to(out), n, m, n, k, parts, w, wb, st),
            "spx_gemm_bf16_nt_tail");
    else
      check(spx_gemm_bf16_auto(route, in(a), a.stride(0), in(b), b.stride(0), to(out), n, m, n, k,
                               m_live.defined() ? m_live.const_data_ptr<int32_t>() : nullptr, parts, w, wb, st),
            "spx_gemm_bf16_auto");
    return out;
  }
  // a b with the rows of b in two matrices (kPairNN); count: as Parted, null where the result is to be stored
  Tensor pair(const Tensor& a, const Tensor& b, const Tensor& b2, int32_t* count) const {
    const int64_t m = a.size(0), k = a.size(1), n = b.size(1);
    TORCH_CHECK_VALUE(b2.defined() && b2.sizes() == b.sizes() && b2.stride(0) == b.stride(0) && 2 * b.size(0) == k,
                      "shape mismatch: a ", a.sizes(), " and two of b ", b.sizes());
    const Tensor out = at::empty({m, n}, a.options());
    check(spx_gemm_bf16_pair(1, in(a), a.stride(0), in(b), in(b2), b.stride(0), to(out), n, m, n, k, parts,
                             ws.defined() ? ws.mutable_data_ptr() : nullptr, ws.defined() ? ws.nbytes() : 0, count, stream_of(a)),
          "spx_gemm_bf16_pair");
    return out;
  }
  // for a launch that adds the parts of a cut product itself
  Parted parted(int64_t route, const Tensor& a, const Tensor& b) const {
    if ((route != kAutoNT && route != kAutoNN) || !ws.defined()) return {(*this)(route, a, b)};
    const int64_t m = a.size(0), k = a.size(1), n = route == kAutoNN ? b.size(1) : b.size(0);
    TORCH_CHECK_VALUE(b.size(route == kAutoNN ? 0 : 1) == k, "shape mismatch: a ", a.sizes(), " b ", b.sizes());
    Parted out{at::empty({m, n}, a.options()), ws.const_data_ptr<float>()};
    check(spx_gemm_bf16_auto_parts(route, in(a), a.stride(0), in(b), b.stride(0), to(out.stored), n, m, n, k, parts,
                                   ws.mutable_data_ptr(), ws.nbytes(), &out.count, stream_of(a)),
          "spx_gemm_bf16_auto_parts");
    return out;
  }
};

}  // namespace

// (route, a, b, m_live, parts, workspace) -> a b^T or a b
PyObject* spx_layer_product(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Args x("product", args, n, 6);
  const int64_t route = x.integer();
  const Tensor &a = x.tensor(), &b = x.tensor(), live = x.maybe();
  const int64_t parts = x.integer();
  const Products product{parts, x.maybe()};
  Unlocked released;
  return wrapped(released, product(route, a, b, live));
  END_HANDLE_TH_ERRORS
}

// Behind the attention: o, residual add + norm, gate/up, SwiGLU, down, residual add + the next norm.
PyObject* spx_layer_tail_forward(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Args x("tail_forward", args, n, 19);
  const Tensor &residual = x.tensor(), &att = x.tensor(), &wo = x.tensor(), &wgu = x.tensor(), &wd = x.tensor(),
               &gain_post = x.tensor(), &gain_next = x.tensor(), slot_gu = x.maybe(), slot_d = x.maybe(),
               slot_next = x.maybe();
  const double eps_post = x.number(), eps_next = x.number();
  const int64_t r_o = x.integer(), r_gu = x.integer(), r_d = x.integer(), parts = x.integer();
  const Products product{parts, x.maybe()};
  const Tensor wu = x.maybe();  // where there is one, wgu is gate's alone
  const int64_t keep = x.integer();  // the gate's and up's outputs are wanted
  Unlocked released;
  const int64_t t = residual.size(0), h = residual.size(1), f = wu.defined() ? wgu.size(0) : wgu.size(0) / 2;
  void* const st = stream_of(residual);
  const Tensor stats = at::empty({2, t}, residual.options().dtype(at::kFloat));
  float* const rstd = floats(stats);
  const Parted o = product.parted(r_o, att, wo);
  const Tensor mid = at::empty({t, h}, residual.options()), z = rows_or_new(slot_gu, t, h, residual);
  add_norm(residual, o, mid, gain_post, z, rstd, eps_post, st);
  const Tensor act = rows_or_new(slot_d, t, f, residual);
  Tensor gu;
  if (r_gu == kGatedNT) {
    TORCH_CHECK_VALUE(wgu.size(1) == h && (!wu.defined() || (wu.sizes() == wgu.sizes() && wu.stride(0) == wgu.stride(0))),
                      "shape mismatch: gate and up of ", h, " inputs");
    if (keep) gu = at::empty({t, 2 * f}, residual.options());
    check(spx_gemm_bf16_gated(in(z), z.stride(0), in(wgu), wu.defined() ? in(wu) : in(wgu) + f * wgu.stride(0), wgu.stride(0),
                              keep ? to(gu) : nullptr, 2 * f, to(act), f, t, f, h, parts,
                              product.ws.defined() ? product.ws.mutable_data_ptr() : nullptr, product.ws.defined() ? product.ws.nbytes() : 0, st),
          "spx_gemm_bf16_gated");
  } else {
    TORCH_CHECK_VALUE(!wu.defined(), "two weights as they lie: the gated product");
    gu = product(r_gu, z, wgu);
    check(spx_swiglu_rows_fwd(in(gu), 2 * f, in(gu) + f, 2 * f, to(act), f, t, f, st), "spx_swiglu_rows_fwd");
  }
  const Parted m = product.parted(r_d, act, wd);
  const Tensor y = at::empty({t, h}, residual.options()), normed = rows_or_new(slot_next, t, h, residual);
  add_norm(mid, m, y, gain_next, normed, rstd + t, eps_next, st);
  return tuple_of(released, {mid, stats, z, gu, act, y, normed});
  END_HANDLE_TH_ERRORS
}

// The way back, from (dy, dn) of (y, normed): -> (gradients of down's, gate/up's and o's outputs, of att).  scratch_*: the
// partial sums of the gains' gradients (accumulate: added to).
PyObject* spx_layer_tail_backward(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Args x("tail_backward", args, n, 24);
  const Tensor dy = x.maybe(), dn = x.maybe();
  const Tensor &mid = x.tensor(), &stats = x.tensor(), &gu = x.tensor(), &y = x.tensor(), &gain_post = x.tensor(),
               &gain_next = x.tensor(), &bo = x.tensor(), &bgu = x.tensor(), &bd = x.tensor(), slot_d = x.maybe(),
               slot_gu = x.maybe(), slot_o = x.maybe(), scratch_post = x.maybe();
  const int64_t acc_post = x.integer();
  const Tensor scratch_next = x.maybe();
  const int64_t acc_next = x.integer();
  const int64_t r_o = x.integer(), r_gu = x.integer(), r_d = x.integer(), parts = x.integer();
  const Products product{parts, x.maybe()};
  const Tensor bu = x.maybe();  // r_gu kPairNN: bgu is gate's alone
  Unlocked released;
  const int64_t t = y.size(0), h = y.size(1), f = gu.size(1) / 2;
  void* const st = stream_of(y);
  const float* const rstd = floats(stats);
  const Tensor dm = rows_or_new(slot_d, t, h, y);
  const Tensor dres = dy.defined() ? grad_rows(dy) : Tensor();
  if (dn.defined()) {
    norm_backward(y, gain_next, grad_rows(dn), dres, rstd + t, dm, scratch_next, acc_next, st);
  } else {
    dm.copy_(dres);
  }
  const Tensor dact = product(r_d, dm, bd), dgu = rows_or_new(slot_gu, t, 2 * f, y);
  check(spx_swiglu_rows_bwd(in(gu), 2 * f, in(gu) + f, 2 * f, in(dact), f, to(dgu), 2 * f, to(dgu) + f, 2 * f, t, f, st),
        "spx_swiglu_rows_bwd");
  Parted dz;
  if (r_gu == kPairNN) {
    dz.stored = product.pair(dgu, bgu, bu, product.ws.defined() ? &dz.count : nullptr);
    if (dz.count > 1) dz.at = product.ws.const_data_ptr<float>();
  } else {
    dz = product.parted(r_gu, dgu, bgu);
  }
  const Tensor da = rows_or_new(slot_o, t, h, y);
  norm_backward(mid, gain_post, dz, dm, rstd, da, scratch_post, acc_post, st);
  return tuple_of(released, {dm, dgu, da, product(r_o, da, bo)});
  END_HANDLE_TH_ERRORS
}

// One TTT step in front of that: q, k, v, rotary embedding, attention over the cache's first (offset + 1) T keys.
PyObject* spx_layer_ttt_forward(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Args x("ttt_forward", args, n, 18);
  const Tensor &xin = x.tensor(), &wqkv = x.tensor(), &pos = x.tensor(), &inv_freq = x.tensor(), &k = x.tensor(),
               &v = x.tensor(), &row_lo = x.tensor(), slot = x.maybe();
  const int64_t hq = x.integer(), hkv = x.integer(), d = x.integer(), offset = x.integer(), step = x.integer();
  const double table_scale = x.number(), scaling = x.number();
  const int64_t route = x.integer(), parts = x.integer();
  const Products product{parts, x.maybe()};
  Unlocked released;
  const int64_t t = xin.size(0), at = offset * t * d;
  TORCH_CHECK_VALUE(k.size(2) >= (offset + 1) * t && row_lo.numel() == t && pos.numel() == t && step == offset,
                    "the layer's cache, mask and positions do not fit step ", offset, " of ", t, " tokens");
  void* const st = stream_of(xin);
  const Tensor qkv = product(route, xin, wqkv);
  const Tensor q = at::empty({1, hq, t, d}, xin.options());
  check(spx_rope_qkv(to(qkv), qkv.size(1), to(q), t * d, to(k) + at, k.stride(1), to(v) + at, v.stride(1),
                     pos.const_data_ptr<int64_t>(), inv_freq.const_data_ptr<float>(), t, hq, hkv, d,
                     2 * inv_freq.numel(), 0, offset, table_scale, st),
        "spx_rope_qkv");
  const Tensor att = rows_or_new(slot, t, hq * d, xin);
  const Tensor lse = attention_forward(q, k, v, Mask{row_lo, {}, {}, {}, t, step}, scaling, att);
  return tuple_of(released, {q, att, lse});
  END_HANDLE_TH_ERRORS
}

// -> (gradient of q, k, v's product, of its input, dk, dv of all keys up to this step).  dk, dv None: this step's node is
// the first of the pass and makes them; otherwise they are added to.
PyObject* spx_layer_ttt_backward(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Args x("ttt_backward", args, n, 21);
  const Tensor &q = x.tensor(), &k = x.tensor(), &v = x.tensor(), &att = x.tensor(), &datt = x.tensor(),
               &lse = x.tensor(), &row_lo = x.tensor();
  Tensor dk = x.maybe(), dv = x.maybe();
  const Tensor slot = x.maybe();
  const Tensor &pos = x.tensor(), &inv_freq = x.tensor();
  const int64_t offset = x.integer();
  const double table_scale = x.number(), scaling = x.number();
  const Tensor& w = x.tensor();
  const int64_t n_qkv = x.integer(), route = x.integer(), parts = x.integer();
  const Products product{parts, x.maybe()};
  const int64_t step = x.integer();
  Unlocked released;
  const int64_t hq = q.size(1), t = q.size(2), d = q.size(3), hkv = k.size(1), keys = (offset + 1) * t, at = offset * t * d;
  void* const st = stream_of(q);
  const bool add = dk.defined();
  if (!add) {
    dk = at::empty({1, hkv, keys, d}, q.options());
    dv = at::empty({1, hkv, keys, d}, q.options());
  }
  TORCH_CHECK_VALUE(dk.size(2) >= keys && dv.size(2) >= keys && k.size(2) >= keys, "gradients of ", keys, " keys");
  const Tensor dq = at::empty_like(q);
  const int64_t nb = spx_ttt_attn_workspace_bytes(t, hq, hkv, d, 1);
  const Tensor ws = bytes(nb, q);
  check((add ? spx_ttt_attn_bwd_accumulate : spx_ttt_attn_bwd)(
            in(q), q.stride(1), in(k), k.stride(1), in(v), v.stride(1), in(att), in(datt), lse.const_data_ptr<float>(),
            row_lo.const_data_ptr<int32_t>(), t, step, hq, hkv, d, scaling, to(dq), dq.stride(1), to(dk), dk.stride(1),
            to(dv), dv.stride(1), ws.mutable_data_ptr(), nb, st),
        "spx_ttt_attn_bwd");
  const Tensor dqkv = rows_or_new(slot, t, n_qkv, q);
  check(spx_rope_qkv(to(dqkv), n_qkv, to(dq), dq.stride(1), to(dk) + at, dk.stride(1), to(dv) + at, dv.stride(1),
                     pos.const_data_ptr<int64_t>(), inv_freq.const_data_ptr<float>(), t, hq, hkv, d,
                     2 * inv_freq.numel(), 1, offset, table_scale, st),
        "spx_rope_qkv");
  return tuple_of(released, {dqkv, product(route, dqkv, w), dk, dv});
  END_HANDLE_TH_ERRORS
}

// Per-head norms, rotation and attention of a layer whose q rows are the last of its key rows or all of them.  kv_column:
// where k begins in a row of kv_tok (v behind it).
PyObject* spx_layer_normed_forward(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Args x("normed_forward", args, n, 22);
  const Tensor &q_tok = x.tensor(), &kv_tok = x.tensor(), &q_pos = x.tensor(), &kv_pos = x.tensor(),
               &inv_freq = x.tensor(), &gain_q = x.tensor(), &gain_k = x.tensor(), slot = x.maybe();
  const int64_t kv_column = x.integer(), hq = x.integer(), hkv = x.integer(), d = x.integer();
  const double table_scale = x.number(), scaling = x.number(), eps_q = x.number(), eps_k = x.number();
  const Tensor &lo = x.tensor(), hi = x.maybe(), blo = x.maybe(), bhi = x.maybe();
  const int64_t T = x.integer(), step = x.integer();
  Unlocked released;
  const int64_t nq = q_tok.size(0), nk = kv_tok.size(0);
  TORCH_CHECK_VALUE(q_pos.numel() == nq && kv_pos.numel() == nk, "positions of ", nq, " and ", nk, " rows");
  void* const st = stream_of(q_tok);
  const Tensor q = at::empty({1, hq, nq, d}, q_tok.options()), kv = at::empty({2, 1, hkv, nk, d}, q_tok.options()),
               rq = at::empty({nq, hq}, q_tok.options().dtype(at::kFloat)),
               rk = at::empty({nk, hkv}, q_tok.options().dtype(at::kFloat));
  const Tensor k = kv.select(0, 0), v = kv.select(0, 1);
  const float* const f = inv_freq.const_data_ptr<float>();
  const spx_head_norm sets[2] = {
      {in(q_tok), q_tok.stride(0), to(q), nq * d, nullptr, 0, q_pos.const_data_ptr<int64_t>(), in(gain_q), floats(rq), nq,
       (int32_t)hq, 0, (float)eps_q, 0, nullptr, 0, nullptr},
      {in(kv_tok) + kv_column, kv_tok.stride(0), to(k), nk * d, to(v), nk * d, kv_pos.const_data_ptr<int64_t>(), in(gain_k),
       floats(rk), nk, (int32_t)hkv, (int32_t)hkv, (float)eps_k, 0, nullptr, 0, nullptr}};
  check(spx_head_norm_rope_sets(sets, 2, f, (int32_t)d, 0, (float)table_scale, st), "spx_head_norm_rope_sets");
  const Tensor att = rows_or_new(slot, nq, hq * d, q_tok);
  const Tensor lse = attention_forward(q, k, v, Mask{lo, hi, blo, bhi, T, step}, scaling, att);
  return tuple_of(released, {q, kv, rq, rk, att, lse});
  END_HANDLE_TH_ERRORS
}

// -> (gradients of the two products).  Without separate k, v (kv_column > 0) both are one.
PyObject* spx_layer_normed_backward(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Args x("normed_backward", args, n, 29);
  const Tensor &q_tok = x.tensor(), &kv_tok = x.tensor(), &q = x.tensor(), &kv = x.tensor(), &rq = x.tensor(),
               &rk = x.tensor(), &att = x.tensor(), &datt = x.tensor(), &lse = x.tensor(), &q_pos = x.tensor(),
               &kv_pos = x.tensor(), &inv_freq = x.tensor(), &gain_q = x.tensor(), &gain_k = x.tensor(),
               slot_q = x.maybe(), slot_kv = x.maybe(), scratch_q = x.maybe();
  const int64_t acc_q = x.integer();
  const Tensor scratch_k = x.maybe();
  const int64_t acc_k = x.integer(), kv_column = x.integer();
  const double table_scale = x.number(), scaling = x.number();
  const Tensor &lo = x.tensor(), hi = x.maybe(), blo = x.maybe(), bhi = x.maybe();
  const int64_t T = x.integer(), step = x.integer();
  Unlocked released;
  const int64_t hq = q.size(1), nq = q.size(2), d = q.size(3), hkv = kv.size(2), nk = kv.size(3);
  void* const st = stream_of(q);
  const auto [dq, dk, dv] = attention_backward(q, kv.select(0, 0), kv.select(0, 1), att, datt, lse,
                                               Mask{lo, hi, blo, bhi, T, step}, scaling);
  const Tensor dq_tok = rows_or_new(slot_q, nq, q_tok.size(1), q),
               dkv_tok = kv_column ? dq_tok : rows_or_new(slot_kv, nk, kv_tok.size(1), q);
  const float* const f = inv_freq.const_data_ptr<float>();
  const spx_head_norm sets[2] = {
      {in(q_tok), q_tok.stride(0), to(dq), nq * d, nullptr, 0, q_pos.const_data_ptr<int64_t>(), in(gain_q), floats(rq), nq,
       (int32_t)hq, 0, 0.f, (int32_t)acc_q, to(dq_tok), dq_tok.stride(0), floats(scratch_q)},
      {in(kv_tok) + kv_column, kv_tok.stride(0), to(dk), nk * d, to(dv), nk * d, kv_pos.const_data_ptr<int64_t>(), in(gain_k),
       floats(rk), nk, (int32_t)hkv, (int32_t)hkv, 0.f, (int32_t)acc_k, to(dkv_tok) + kv_column, dkv_tok.stride(0),
       floats(scratch_k)}};
  check(spx_head_norm_rope_bwd_sets(sets, 2, f, (int32_t)d, 0, (float)table_scale, st), "spx_head_norm_rope_bwd_sets");
  return tuple_of(released, {dq_tok, dkv_tok});
  END_HANDLE_TH_ERRORS
}

// The weight gradient a^T b: (a [T, M], b [T, N], out or None, accumulate, fp32, workspace or None) -> [M, N]
PyObject* spx_layer_product_tn(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Args x("product_tn", args, n, 6);
  const Tensor &a = x.tensor(), &b = x.tensor();
  Tensor out = x.maybe();
  const int64_t accumulate = x.integer(), f32 = x.integer();
  const Tensor ws = x.maybe();
  Unlocked released;
  const int64_t t = a.size(0), m = a.size(1), cols = b.size(1);
  if (!out.defined()) out = at::empty({m, cols}, a.options().dtype(f32 ? at::kFloat : at::kBFloat16));
  check(spx_gemm_bf16_tn_auto(in(a), a.stride(0), in(b), b.stride(0), out.mutable_data_ptr(), out.stride(0), m, cols, t, f32,
                              accumulate, ws.defined() ? ws.mutable_data_ptr() : nullptr,
                              ws.defined() ? (int64_t)ws.nbytes() : 0, stream_of(a)),
        "spx_gemm_bf16_tn_auto");
  return wrapped(released, out);
  END_HANDLE_TH_ERRORS
}

// Weight gradients in one launch: (fp32, workspace or None, then for each a [T, M], b [T, N], out [M, N] or None)
// -> the results
PyObject* spx_layer_products_tn(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TORCH_CHECK_TYPE(n >= 5 && n % 3 == 2 && n <= 26, "products_tn takes three arguments for each of 1 .. 8 products, and two");
  Args x("products_tn", args, n, n);
  const int64_t f32 = x.integer();
  const Tensor ws = x.maybe();
  const int count = (int)(n / 3);
  Tensor a[8], b[8], out[8];
  for (int i = 0; i < count; ++i) {
    a[i] = x.tensor();
    b[i] = x.tensor();
    out[i] = x.maybe();
    TORCH_CHECK_VALUE(a[i].dim() == 2 && b[i].dim() == 2 && a[i].size(0) == b[i].size(0) && a[i].stride(1) == 1 && b[i].stride(1) == 1 &&
                          a[i].scalar_type() == at::kBFloat16 && b[i].scalar_type() == at::kBFloat16 && a[i].device() == a[0].device() &&
                          b[i].device() == a[0].device(),
                      "bf16 operands [T, M], [T, N] with contiguous rows, on one device");
    TORCH_CHECK_VALUE(!out[i].defined() || (out[i].dim() == 2 && out[i].size(0) == a[i].size(1) && out[i].size(1) == b[i].size(1) &&
                                            out[i].stride(1) == 1 && out[i].scalar_type() == (f32 ? at::kFloat : at::kBFloat16) &&
                                            out[i].device() == a[0].device()),
                      "out does not fit its product");
  }
  Unlocked released;
  spx_tn_product list[8];
  for (int i = 0; i < count; ++i) {
    if (!out[i].defined())
      out[i] = at::empty({a[i].size(1), b[i].size(1)}, a[i].options().dtype(f32 ? at::kFloat : at::kBFloat16).requires_grad(false));
    list[i] = {in(a[i]), a[i].stride(0), in(b[i]), b[i].stride(0), out[i].mutable_data_ptr(), out[i].stride(0),
               a[i].size(1), b[i].size(1), a[i].size(0)};
  }
  check(spx_gemm_bf16_tn_list(list, count, (int)f32, ws.defined() ? ws.mutable_data_ptr() : nullptr,
                              ws.defined() ? (int64_t)ws.nbytes() : 0, stream_of(a[0])),
        "spx_gemm_bf16_tn_list");
  released.lock();
  PyObject* const all = PyTuple_New(count);
  for (int i = 0; i < count; ++i) PyTuple_SET_ITEM(all, i, THPVariable_Wrap(out[i]));
  return all;
  END_HANDLE_TH_ERRORS
}

// One TTT step's loss over bf16 logits in one read of the rows, with its masked mean: (op, logits, targets or None, known
// lse_t, known argmax_t or None, mask, its kind, prev or None, its kind, acceptance counts or None (made and cleared here),
// loss so far or None, step weight, term factor, scalars [8] or None: no mean) -> (total, row losses, argmax_draft,
// argmax_target, lse_target, packed logits gradient, row map, live rows, row weights, rows by slot)
PyObject* spx_layer_loss_step(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Args x("loss_step", args, n, 14);
  const int64_t op = x.integer();
  const Tensor &logits = x.tensor(), y = x.maybe(), known_lse = x.maybe(), known_arg = x.maybe(), &mask = x.tensor();
  const int64_t mask_kind = x.integer();
  const Tensor prev = x.maybe();
  const int64_t prev_kind = x.integer();
  const Tensor given = x.maybe(), total_in = x.maybe();
  const double weight = x.number(), factor = x.number();
  const Tensor out = x.maybe();
  Unlocked released;
  const int64_t rows = logits.size(0), vocab = logits.size(1);
  const bool known = known_lse.defined();
  void* const st = stream_of(logits);
  const auto i32 = logits.options().dtype(at::kInt), f32 = logits.options().dtype(at::kFloat);
  const Tensor map = at::empty({2 * rows + 1}, i32), arg = at::empty({2 * rows + 3}, i32), stats = at::empty({5 * rows}, f32),
               packed = at::empty({rows, vocab}, logits.options()), total = at::empty({}, f32);
  int32_t* const row_map = map.mutable_data_ptr<int32_t>();  // the map, the count, the rows by slot
  int32_t* const am = arg.mutable_data_ptr<int32_t>();
  int32_t* const counts = given.defined() ? given.mutable_data_ptr<int32_t>() : am + 2 * rows;
  float* const s = floats(stats);  // loss, lse_draft, lse_target, extra, row weights
  float* const lse_t = known ? known_lse.mutable_data_ptr<float>() : s + 2 * rows;
  int32_t* const am_t = known ? known_arg.mutable_data_ptr<int32_t>() : am + rows;
  check(spx_mask_row_lists(mask.const_data_ptr(), mask_kind, rows, row_map, row_map + rows, row_map + rows + 1,
                           given.defined() ? nullptr : counts, st),
        "spx_mask_row_lists");
  check(spx_vocab_loss_step_fwd_grad(op, in(logits), logits.stride(0), y.defined() ? in(y) : nullptr,
                                     y.defined() ? y.stride(0) : 0, rows, vocab, s, s + rows, lse_t, s + 3 * rows, am, am_t,
                                     known, mask.const_data_ptr(), mask_kind,
                                     prev.defined() ? prev.mutable_data_ptr() : nullptr, prev_kind, counts, row_map,
                                     to(packed), vocab, st),
        "spx_vocab_loss_step_fwd_grad");
  if (out.defined())
    check(spx_ttt_step_total(s, am, am_t, mask.const_data_ptr(), mask_kind, nullptr, 0, rows, weight, counts, factor,
                             total_in.defined() ? total_in.const_data_ptr<float>() : nullptr, floats(total),
                             floats(out), s + 4 * rows, st),
          "spx_ttt_step_total");
  return tuple_of(released, {total, stats.narrow(0, 0, rows), arg.narrow(0, 0, rows),
                             known ? known_arg : arg.narrow(0, rows, rows),
                             known ? known_lse : stats.narrow(0, 2 * rows, rows), packed, map.narrow(0, 0, rows),
                             map.narrow(0, rows, 1), stats.narrow(0, 4 * rows, rows), map.narrow(0, rows + 1, rows)});
  END_HANDLE_TH_ERRORS
}

// The same for a loss of several terms (spx_vocab_loss_terms_fwd_grad); d2t: the targets are full-vocabulary rows, gathered
// first by the pass that leaves their statistics behind
PyObject* spx_layer_loss_terms(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Args x("loss_terms", args, n, 18);
  const int32_t terms = (int32_t)x.integer();
  float weights[5];
  for (float& w : weights) w = (float)x.number();
  const Tensor &logits = x.tensor(), &targets = x.tensor();
  const Tensor d2t = x.maybe(), known_lse = x.maybe(), known_arg = x.maybe(), &mask = x.tensor();
  const int64_t mask_kind = x.integer();
  const Tensor prev = x.maybe();
  const int64_t prev_kind = x.integer();
  const Tensor total_in = x.maybe();
  const double weight = x.number();
  const Tensor& out = x.tensor();
  Unlocked released;
  const int64_t rows = logits.size(0), vocab = logits.size(1);
  bool known = known_lse.defined();
  void* const st = stream_of(logits);
  const auto i32 = logits.options().dtype(at::kInt), f32 = logits.options().dtype(at::kFloat);
  const Tensor map = at::empty({2 * rows + 1}, i32), arg = at::empty({2 * rows + 3}, i32), stats = at::empty({9 * rows}, f32),
               packed = at::empty({rows, vocab}, logits.options()), total = at::empty({}, f32);
  int32_t* const row_map = map.mutable_data_ptr<int32_t>();
  int32_t* const am = arg.mutable_data_ptr<int32_t>();
  int32_t* const counts = am + 2 * rows;
  float* const s = floats(stats);  // lse_draft, lse_target, row weights, one more, up to five terms' losses
  float* const lse_t = known ? known_lse.mutable_data_ptr<float>() : s + rows;
  int32_t* const am_t = known ? known_arg.mutable_data_ptr<int32_t>() : am + rows;
  check(spx_mask_row_lists(mask.const_data_ptr(), mask_kind, rows, row_map, row_map + rows, row_map + rows + 1, counts, st),
        "spx_mask_row_lists");
  Tensor gathered;
  if (d2t.defined()) {
    gathered = at::empty({rows, vocab}, logits.options());
    check(spx_vocab_loss_step_fwd(SPX_LOSS_KL, in(logits), logits.stride(0), in(targets), targets.stride(0),
                                  d2t.const_data_ptr<int64_t>(), targets.size(1), to(gathered), vocab, rows, vocab,
                                  SPX_DTYPE_BF16, s + 4 * rows, s, lse_t, s + 3 * rows, am, am_t, 0, nullptr, 0, nullptr, 0,
                                  nullptr, st),
          "spx_vocab_loss_step_fwd");
    known = true;
  }
  const Tensor& y = gathered.defined() ? gathered : targets;
  check(spx_vocab_loss_terms_fwd_grad(terms, weights, in(logits), logits.stride(0), in(y), y.stride(0), rows, vocab,
                                      s + 4 * rows, s, lse_t, am, am_t, known, mask.const_data_ptr(), mask_kind,
                                      prev.defined() ? prev.mutable_data_ptr() : nullptr, prev_kind, counts, row_map,
                                      to(packed), vocab, st),
        "spx_vocab_loss_terms_fwd_grad");
  check(spx_ttt_step_terms(terms, weights, s + 4 * rows, mask.const_data_ptr(), mask_kind, rows, weight, counts,
                           total_in.defined() ? total_in.const_data_ptr<float>() : nullptr, floats(total), floats(out),
                           s + 2 * rows, st),
        "spx_ttt_step_terms");
  const bool given = known_lse.defined();
  return tuple_of(released, {total, arg.narrow(0, 0, rows), given ? known_arg : arg.narrow(0, rows, rows),
                             given ? known_lse : stats.narrow(0, rows, rows), packed, map.narrow(0, 0, rows),
                             map.narrow(0, rows, 1), stats.narrow(0, 2 * rows, rows), map.narrow(0, rows + 1, rows), y});
  END_HANDLE_TH_ERRORS
}

// The loss of all steps of a TTT loop (spx_loss_steps_*).  What its launches share lies in two buffers:
struct LossSteps {
  int64_t T, steps;
  int32_t terms = 0;  // a set of ops with their weights (0: one loss)
  float weights[5];
  int32_t *row_map, *live, *slots, *ticket, *full, *row_slot, *slot_row;
  float *inv, *mask_sum, *loss, *row_weight, *partials;
  static int64_t ints(int64_t T, int64_t steps) { return T + 3 + steps + 2 * steps * T; }
  int64_t losses() const { return (terms ? __builtin_popcount(terms) : 1) * steps * T; }
  int64_t all_floats() const { return 2 * steps + steps * T + losses() + spx_loss_steps_partials(T, (int32_t)steps, terms); }
  LossSteps(int64_t T_, int64_t steps_, PyObject* term_weights) : T(T_), steps(steps_) {  // None or five numbers, 0: no such term
    if (term_weights == Py_None) return;
    TORCH_CHECK_TYPE(PyTuple_Check(term_weights) && PyTuple_GET_SIZE(term_weights) == 5, "five term weights or None");
    for (int op = 0; op < 5; ++op) {
      PyObject* const w = PyTuple_GET_ITEM(term_weights, op);
      weights[op] = 0.f;
      if (w == Py_None) continue;
      terms |= 1 << op;
      weights[op] = (float)PyFloat_AsDouble(w);
      if (PyErr_Occurred()) throw python_error();
    }
  }
  void bind(const Tensor& i, const Tensor& f) {
    TORCH_CHECK_VALUE(i.scalar_type() == at::kInt && f.scalar_type() == at::kFloat && i.is_contiguous() && f.is_contiguous() &&
                          i.numel() == ints(T, steps) && f.numel() == all_floats(),
                      "the buffers of loss_steps_begin for ", T, " rows and ", steps, " steps");
    row_map = i.mutable_data_ptr<int32_t>();
    live = row_map + T; slots = live + 1; ticket = slots + 1; full = ticket + 1; row_slot = full + steps;
    slot_row = row_slot + steps * T;
    inv = f.mutable_data_ptr<float>();
    mask_sum = inv + steps; row_weight = mask_sum + steps; loss = row_weight + steps * T; partials = loss + losses();
  }
};

// (mask, its kind, term weights or None, the steps' weights ..) -> (integers, floats; views: live slots, row -> slot, slot -> row, row weights)
PyObject* spx_layer_loss_steps_begin(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  const int64_t steps = n - 3;
  TORCH_CHECK_TYPE(steps >= 1 && steps <= SPX_LOSS_STEPS_MAX, "loss_steps_begin takes 1 .. 32 step weights");
  Args x("loss_steps_begin", args, n, n);
  const Tensor& mask = x.tensor();
  const int64_t kind = x.integer(), T = mask.numel();
  LossSteps s(T, steps, *x.at++);
  float weights[SPX_LOSS_STEPS_MAX];
  for (int64_t k = 0; k < steps; ++k) weights[k] = (float)x.number();
  Unlocked released;
  const Tensor i = at::empty({LossSteps::ints(T, steps)}, mask.options().dtype(at::kInt).requires_grad(false)),
               f = at::empty({s.all_floats()}, mask.options().dtype(at::kFloat).requires_grad(false));
  s.bind(i, f);
  check(spx_loss_steps_mask(mask.const_data_ptr(), kind, T, (int32_t)steps, weights, s.row_map, s.live, s.inv, s.mask_sum,
                            s.full, s.ticket, stream_of(mask)),
        "spx_loss_steps_mask");
  const int64_t lists = s.row_slot - s.row_map, w = s.row_weight - s.inv;
  return tuple_of(released, {i, f, i.narrow(0, T + 1, 1), i.narrow(0, lists, steps * T),
                             i.narrow(0, lists + steps * T, steps * T), f.narrow(0, w, steps * T)});
  END_HANDLE_TH_ERRORS
}

// (op, term weights or None, masked rows of step 0 formed?, mask, its kind, targets or None, their arg-max or None, integers, floats, tokens [steps, T], hits [steps, T], packed
// gradient [steps * T, vocab] or None, steps, first step, logits [T, vocab] of this and the following steps ..)
PyObject* spx_layer_loss_steps_pass(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  const int64_t here = n - 14;
  TORCH_CHECK_TYPE(here >= 1 && here <= SPX_LOSS_STEPS_MAX, "loss_steps_pass takes the logits of 1 .. 32 steps");
  Args x("loss_steps_pass", args, n, n);
  const int64_t op = x.integer();
  PyObject* const term_weights = *x.at++;
  const int64_t masked_first = x.integer();
  const Tensor& mask = x.tensor();
  const int64_t kind = x.integer();
  const Tensor y = x.maybe(), known = x.maybe();
  const Tensor &i = x.tensor(), &f = x.tensor(), &tokens = x.tensor(), &hits = x.tensor();
  const Tensor packed = x.maybe();
  const int64_t steps = x.integer(), first = x.integer();
  const void* logits[SPX_LOSS_STEPS_MAX];
  int64_t vocab = 0, ld = 0;
  const int64_t T = mask.numel();
  for (int64_t k = 0; k < here; ++k) {
    const Tensor& l = x.tensor();
    if (k == 0) { vocab = l.size(1); ld = l.stride(0); }
    TORCH_CHECK_VALUE(l.dim() == 2 && l.size(0) == T && l.size(1) == vocab && l.stride(0) == ld && l.stride(1) == 1 &&
                          l.scalar_type() == at::kBFloat16 && l.device() == mask.device(),
                      "bf16 logits [rows, vocab], all alike");
    logits[k] = l.const_data_ptr();
  }
  TORCH_CHECK_VALUE((!y.defined() || (y.size(0) == T && y.size(1) == vocab && y.stride(1) == 1 && y.scalar_type() == at::kBFloat16)) &&
                        (!known.defined() || (known.numel() == T && known.is_contiguous() && known.scalar_type() == at::kInt)) &&
                        tokens.numel() == steps * T && hits.numel() == steps * T && tokens.scalar_type() == at::kLong &&
                        hits.scalar_type() == at::kByte && tokens.is_contiguous() && hits.is_contiguous() &&
                        (!packed.defined() || (packed.numel() == steps * T * vocab && packed.is_contiguous() &&
                                               packed.scalar_type() == at::kBFloat16)),
                    "targets, their arg-max, tokens, hits or gradient do not fit the logits");
  LossSteps s(T, steps, term_weights);
  s.bind(i, f);
  Unlocked released;
  check(spx_loss_steps_pass((int)op, s.terms, s.weights, logits, ld, y.defined() ? in(y) : nullptr, y.defined() ? y.stride(0) : 0,
                            known.defined() ? known.const_data_ptr<int32_t>() : nullptr, T, vocab, (int32_t)steps,
                            (int32_t)first, (int32_t)(first + here), masked_first != 0, mask.const_data_ptr(), kind, s.inv, s.row_map, s.live,
                            s.loss, tokens.mutable_data_ptr<int64_t>(), hits.mutable_data_ptr<uint8_t>(), s.row_slot,
                            s.slot_row, s.slots, s.row_weight, packed.defined() ? to(packed) : nullptr, vocab,
                            stream_of(mask)),
        "spx_loss_steps_pass");
  released.lock();
  Py_RETURN_NONE;
  END_HANDLE_TH_ERRORS
}

// (term weights or None, mask, its kind, prev or None, its kind, integers, floats, hits, steps, term factor) -> (scalars
// [steps, 8], of several terms [steps, 18], loss)
PyObject* spx_layer_loss_steps_end(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Args x("loss_steps_end", args, n, 10);
  PyObject* const term_weights = *x.at++;
  const Tensor& mask = x.tensor();
  const int64_t kind = x.integer();
  const Tensor prev = x.maybe();
  const int64_t prev_kind = x.integer();
  const Tensor &i = x.tensor(), &f = x.tensor(), &hits = x.tensor();
  const int64_t steps = x.integer();
  const double factor = x.number();
  const int64_t T = mask.numel();
  TORCH_CHECK_VALUE(hits.numel() == steps * T && (!prev.defined() || (prev.numel() >= T && prev.is_contiguous())),
                    "hits or prev do not fit the mask");
  LossSteps s(T, steps, term_weights);
  s.bind(i, f);
  Unlocked released;
  const Tensor out = at::empty({steps, s.terms ? 18 : 8}, f.options()), total = at::empty({}, f.options());
  check(spx_loss_steps_total(s.loss, hits.const_data_ptr<uint8_t>(), mask.const_data_ptr(), kind,
                             prev.defined() ? prev.mutable_data_ptr() : nullptr, prev_kind, T, (int32_t)steps, (float)factor,
                             s.terms, s.weights, s.inv, s.mask_sum, s.full, s.partials, s.ticket, floats(out), floats(total), stream_of(mask)),
        "spx_loss_steps_total");
  return tuple_of(released, {out, total});
  END_HANDLE_TH_ERRORS
}

// The row-wise concatenation of one to four matrices as one bf16 matrix
PyObject* spx_layer_cat_bf16(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TORCH_CHECK_TYPE(n >= 1 && n <= 8, "cat_bf16 takes one to eight tensors");
  Args x("cat_bf16", args, n, n);
  const void* src[8];
  int64_t elements[8], rows = 0;
  int32_t f32[8];
  Tensor first;
  for (Py_ssize_t i = 0; i < n; ++i) {
    const Tensor& t = x.tensor();
    if (i == 0) first = t;
    TORCH_CHECK_VALUE(t.is_contiguous() && t.dim() >= 1 && t.sizes().slice(1) == first.sizes().slice(1) &&
                          t.device() == first.device() &&
                          (t.scalar_type() == at::kFloat || t.scalar_type() == at::kBFloat16),
                      "contiguous bf16 or fp32 matrices of one width");
    src[i] = t.const_data_ptr();
    elements[i] = t.numel();
    f32[i] = t.scalar_type() == at::kFloat;
    rows += t.size(0);
  }
  Unlocked released;
  auto shape = first.sizes().vec();
  shape[0] = rows;
  const Tensor out = at::empty(shape, first.options().dtype(at::kBFloat16).requires_grad(false));
  check(spx_cat_bf16(src, elements, f32, n, out.mutable_data_ptr(), stream_of(first)), "spx_cat_bf16");
  return wrapped(released, out);
  END_HANDLE_TH_ERRORS
}

// (partial sums, slots, H, fp32 out?) per gain -> a tuple of their sums [H], sixteen gains to a launch
PyObject* spx_layer_gain_sums(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TORCH_CHECK_TYPE(n >= 4 && n % 4 == 0, "gain_sums takes four arguments for every gain");
  const int64_t gains = n / 4;
  Args x("gain_sums", args, n, n);
  std::vector<Tensor> part(gains), out(gains);
  std::vector<const float*> from(gains);
  std::vector<void*> into(gains);
  std::vector<int64_t> slots(gains), h(gains);
  std::vector<int32_t> f32(gains);
  for (int64_t i = 0; i < gains; ++i) {
    part[i] = x.tensor();
    slots[i] = x.integer();
    h[i] = x.integer();
    f32[i] = x.integer() != 0;
    TORCH_CHECK_VALUE(part[i].scalar_type() == at::kFloat && part[i].is_contiguous() && slots[i] > 0 && h[i] > 0 &&
                          part[i].numel() >= slots[i] * h[i] && part[i].device() == part[0].device(),
                      "contiguous fp32 partial sums of slots x H, on one device");
  }
  Unlocked released;
  for (int64_t i = 0; i < gains; ++i) {
    out[i] = at::empty({h[i]}, part[i].options().dtype(f32[i] ? at::kFloat : at::kBFloat16).requires_grad(false));
    from[i] = part[i].const_data_ptr<float>();
    into[i] = out[i].mutable_data_ptr();
  }
  for (int64_t i = 0; i < gains; i += 16)
    check(spx_rmsnorm_dweights(&from[i], &slots[i], &h[i], &into[i], &f32[i], (int32_t)std::min<int64_t>(16, gains - i),
                               stream_of(part[0])), "spx_rmsnorm_dweights");
  released.lock();
  PyObject* const all = PyTuple_New(gains);
  for (int64_t i = 0; i < gains; ++i) PyTuple_SET_ITEM(all, i, THPVariable_Wrap(out[i]));
  return all;
  END_HANDLE_TH_ERRORS
}
