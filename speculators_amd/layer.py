"""A draft decoder layer -- one TTT step of it, or one pass -- as ONE autograd node.

The layer (models/eagle3/model_definitions.py:14-110) is nine launches forward and eleven backward; as
eight nodes of their own they cost more host time (a node's forward and backward 20 us, and the views,
slot look-ups and gradient checks between them) than the kernels take up to a thousand tokens: at 512
tokens of the 1B shape a step of forward and backward was 0.61 ms of host time, 0.33 ms as one node.
The kernels, their order and their buffers (``weights.Staged`` slots, the layer's K / V cache) are those of the
layer put together from its parts, with one difference: the anchored-block layer's k and v are one product.

Whatever the backward reads beside the activations -- the compute weights, which for bf16 parameters are the
parameters themselves, positions, rotary frequencies, mask bounds -- is saved with the node, so that autograd
refuses a backward after one of them was changed in place.
"""

from __future__ import annotations

import torch
from torch.nn.modules import module as M

from . import _lib
from . import attention as A
from . import fused_ops as FO
from . import gemm


def passed_by(cls):
    """Class decorator: modules of ``cls`` are not called where their layer runs as one node."""
    cls.forward_as_written = cls.forward
    return cls


def untouched(*modules) -> bool:
    """Whether calling each of these modules would be its ``passed_by`` class's own ``forward`` and nothing else: no hook
    on it or on every module, no other class, method or compiled call in its place."""
    return not M._has_any_global_hook() and all(
        type(m).forward is getattr(type(m), "forward_as_written", None) and "forward" not in m.__dict__
        and m._compiled_call_impl is None and not (m._forward_hooks or m._forward_pre_hooks or m._backward_hooks
                                                   or m._backward_pre_hooks) for m in modules)


class LayerStep:
    """What a step needs besides its differentiable inputs."""

    __slots__ = ("first", "wqkv", "wo", "wgu", "wd", "eps_in", "eps_post", "eps_next", "hq", "hkv", "d", "scaling",
                 "offset", "positions", "inv_freq", "cache", "mask", "slots", "pair")

    def __init__(self, first, wqkv, wo, wgu, wd, eps, heads, scaling, offset, positions, inv_freq, cache, mask):
        self.first = first
        self.wqkv, self.wo, self.wgu, self.wd = wqkv, wo, wgu, wd
        self.eps_in, self.eps_post, self.eps_next = eps
        self.hq, self.hkv, self.d = heads
        self.scaling, self.offset, self.positions, self.inv_freq = scaling, offset, positions, inv_freq
        self.cache, self.mask = cache, mask
        self.slots = (None,) * 5

    def take_slots(self, t: int, next_staged=None):
        """Where the inputs of the four products (and the next layer's first one) go: the staged weights'
        input buffers.  Asked for outside the node, where grad mode still says whether there is a graph."""
        self.slots = (self.wqkv.x_slot(t) if self.first else None, self.wo.x_slot(t), self.wgu.x_slot(t),
                      self.wd.x_slot(t), next_staged.x_slot(t) if next_staged is not None else None)

    def constants(self):
        """What the backward reads beside activations and gains, to be saved with the node."""
        return (self.positions, self.inv_freq, self.mask.row_lo, self.wqkv.w, self.wo.w, self.wd.w, *_gate_up(self))


def _gate_up(s):
    """The weight of the gate and up projections as the products read it."""
    return (s.wgu.w,) if s.pair is None else s.wgu.pieces


def _rows(t, rows, cols, device):
    return t if t is not None else torch.empty(rows, cols, device=device, dtype=torch.bfloat16)


def _flat(x):
    x2 = x.reshape(-1, x.shape[-1])
    return x2 if x2.stride(1) == 1 else x2.contiguous()


def step_forward(s: LayerStep, a, b, gain_a, gain_b, gain_post, gain_next, keep: bool = True):
    """``(y, normed, saved)``: the layer's output ``[T, H]``, the next norm of it, and what the backward reads (``keep``: if there is
    one)."""
    a2, b2 = _flat(a), _flat(b)
    t, h = a2.shape
    dev = a2.device
    st = _lib.stream_ptr(dev)
    slot_qkv, slot_o, slot_gu, slot_d, slot_next = s.slots
    if s.first:  # a: embeds, b: hidden
        rstd_in = torch.empty(2, t, device=dev, dtype=torch.float32)
        xin = _rows(slot_qkv, t, 2 * h, dev)
        FO.pair_norm_rows(a2, b2, gain_a, gain_b, s.eps_in, xin, rstd_in)
        residual = b2
    else:  # a: the residual stream, b: its norm
        rstd_in, xin, residual = None, b2, a2
    cache, mask = s.cache, s.mask
    route, ws = gemm.forward_route(t, s.wqkv)
    q, att, lse = _lib.native().ttt_forward(
        xin, s.wqkv.w, s.positions, s.inv_freq, cache.k, cache.v, mask.row_lo, slot_o, s.hq, s.hkv, s.d, s.offset,
        mask.ttt_step, FO.table_scale_of(s.inv_freq), s.scaling, route, gemm.TAIL_PARTS, gemm.workspace_for(dev, ws))
    y, normed, tail = _tail_forward(s, residual, att, gain_post, gain_next, slot_gu, slot_d, slot_next, keep)
    return y, normed, (a2, b2, rstd_in, xin, q, att, lse, *tail)


def _tail_forward(s, residual, att, gain_post, gain_next, slot_gu, slot_d, slot_next, keep):
    """What follows the attention: output projection, residual add and norm, MLP, residual add and the norm
    that reads the layer's output."""
    t = residual.shape[0]
    s.pair = gemm.pair_routes(t, s.wgu)
    r_o, r_d = gemm.forward_route(t, s.wo), gemm.forward_route(t, s.wd)
    ws = gemm.gated(t, s.wgu, s.pair)
    if ws is not None:
        r_gu = gemm.GATED_NT, ws
    else:  # (nothing else reads two weights as they lie)
        s.pair, r_gu = None, gemm.forward_route(t, s.wgu)
    routes, sizes = zip(r_o, r_gu, r_d)
    gate, *up = _gate_up(s)
    *tail, y, normed = _lib.native().tail_forward(
        residual, att, s.wo.w, gate, s.wd.w, gain_post, gain_next, slot_gu, slot_d, slot_next, s.eps_post, s.eps_next,
        *routes, gemm.TAIL_PARTS, gemm.workspace_for(residual.device, *sizes), *(up or (None,)),
        int(keep))
    return y, normed, (*tail, y)


class _GainSum:
    """Where one use of a gain leaves the partial sums of its gradient, and what its node returns for it."""

    __slots__ = ("grads", "scratch", "acc", "own")

    def __init__(self, grads, needed: bool, rows: int, h: int, device):
        self.grads, self.scratch, self.acc, self.own = grads, None, 0, False
        if not needed:
            self.grads = None
            return
        shared = grads.target(rows, h, device) if grads is not None else None
        if shared is not None:
            self.scratch, self.acc = shared
        else:
            slots = int(_lib.native().spx_rmsnorm_bwd_slots(rows, h))
            self.scratch, self.own = torch.empty(slots, h, device=device, dtype=torch.float32), True

    def result(self):
        if self.scratch is None:
            return None
        dev = self.scratch.device
        if not self.own:
            return self.grads.mark(dev)
        slots, h = self.scratch.shape
        dw = torch.empty(h, device=dev, dtype=torch.bfloat16)
        _lib.call("spx_rmsnorm_dweight", self.scratch, slots, h, dw, _lib.stream_ptr(dev))
        return dw


def _tail_backward(s, dy, dn, att, tail, gain_post, gain_next, grads_post, grads_next, needs, taken):
    """``(gradient of the residual stream in front of the attention, gradient of att, of the two gains, tokens of
    wo, wgu, wd)``."""
    mid, stats, z, gu, act, y = tail
    slot_o, slot_gu, slot_d = taken
    t, h = y.shape
    dev = y.device
    nxt = _GainSum(grads_next, needs[1] and dn is not None, t, h, dev)
    post = _GainSum(grads_post, needs[0], t, h, dev)
    if s.pair is None:
        r_gu, up = gemm.backward_route(t, s.wgu), None
    else:
        gate, up = s.wgu.pieces
        r_gu = gemm.PAIR_NN, s.pair, gate
    routes, sizes, right = zip(gemm.backward_route(t, s.wo), r_gu, gemm.backward_route(t, s.wd))
    dm, dgu, da, datt = _lib.native().tail_backward(
        dy, dn, mid, stats, gu, y, gain_post, gain_next, *right, s.wd.dy_slot(slot_d, t), s.wgu.dy_slot(slot_gu, t),
        s.wo.dy_slot(slot_o, t), post.scratch, post.acc, nxt.scratch, nxt.acc, *routes, gemm.TAIL_PARTS,
        gemm.workspace_for(dev, *sizes), up)
    tok_d, tok_gu, tok_o = s.wd.defer(slot_d, dm, act), s.wgu.defer(slot_gu, dgu, z), s.wo.defer(slot_o, da, att)
    return da, datt, post.result(), nxt.result(), tok_o, tok_gu, tok_d


class _LayerStep(torch.autograd.Function):
    """``(a, b, gains, tokens) -> (y, norm(y))``; ``a, b``: embeddings and hidden state for the first layer,
    residual stream and its norm for the others.  The keys and values of earlier steps are no edges of the
    node: every earlier step's node runs after this one in a backward pass (the hidden state links them), and
    the gradients of the shared cache meet in its ``_CacheGrads``."""

    @staticmethod
    def forward(ctx, s: LayerStep, a, b, gain_a, gain_b, gain_post, gain_next, *_tokens):
        shape = a.shape
        y, normed, saved = step_forward(s, a, b, gain_a, gain_b, gain_post, gain_next)
        _, _, _, xin, _, att, _, _, _, z, _, act, _ = saved
        ctx.taken = (s.wqkv.take(xin), s.wo.take(att), s.wgu.take(z), s.wd.take(act))
        ctx.gain_grads = tuple(getattr(g, "spx_gain_grads", None) for g in (gain_a, gain_b, gain_post, gain_next))
        ctx.step = s
        ctx.shape = shape
        ctx.save_for_backward(*saved, gain_a, gain_b, gain_post, gain_next, *s.constants())
        ctx.set_materialize_grads(False)
        return y.view(shape), normed.view(shape)

    @staticmethod
    def backward(ctx, dy, dn):
        if dy is None and dn is None:
            return (None,) * 11
        # (the weights come back for autograd's check alone: the products take them from the staged weights)
        (a2, b2, rstd_in, xin, q, att, lse, mid, stats, z, gu, act, y,
         gain_a, gain_b, gain_post, gain_next, positions, inv_freq, row_lo, *_weights) = ctx.saved_tensors
        s = ctx.step
        needs = ctx.needs_input_grad
        t = y.shape[0]
        slot_qkv = ctx.taken[0]
        grads_a, grads_b, grads_post, grads_next = ctx.gain_grads
        da, datt, d_post, d_next, tok_o, tok_gu, tok_d = _tail_backward(
            s, dy, dn, att, (mid, stats, z, gu, act, y), gain_post, gain_next, grads_post, grads_next, needs[5:7],
            ctx.taken[1:])
        n, cache, mask = s.offset + 1, s.cache, s.mask
        dk, dv = cache.grads.enter(n)
        route, ws, right = gemm.backward_route(t, s.wqkv)
        dqkv, dxin, dk, dv = _lib.native().ttt_backward(
            q, cache.k, cache.v, att, datt, lse, row_lo, dk, dv, s.wqkv.dy_slot(slot_qkv, t), positions, inv_freq,
            s.offset, FO.table_scale_of(s.inv_freq), s.scaling, right, s.wqkv.w.shape[0], route, gemm.TAIL_PARTS,
            gemm.workspace_for(q.device, ws), mask.ttt_step)
        cache.grads.leave(n, dk, dv)
        tok_qkv = s.wqkv.defer(slot_qkv, dqkv, xin)
        d_gain_a = d_gain_b = None
        if s.first:
            d_a, d_b, d_gain_a, d_gain_b = FO.pair_norm_rows_backward(
                a2, b2, gain_a, gain_b, dxin, da, rstd_in, (grads_a, grads_b), (needs[1], needs[2], needs[3], needs[4]))
        else:
            d_a, d_b = da, dxin
        if d_a is not None:
            d_a = d_a.view(ctx.shape)
        if d_b is not None:
            d_b = d_b.view(ctx.shape)
        return (None, d_a, d_b, d_gain_a, d_gain_b, d_post, d_next, tok_qkv, tok_o, tok_gu, tok_d)


def run(s: LayerStep, a, b, gain_a, gain_b, gain_post, gain_next):
    """``(y, normed)`` of one step, as one node where there is a graph (every product's weight then trains)."""
    if torch.is_grad_enabled():
        return _LayerStep.apply(s, a, b, gain_a, gain_b, gain_post, gain_next, s.wqkv.token, s.wo.token, s.wgu.token,
                                s.wd.token)
    y, normed, _ = step_forward(s, a, b, gain_a, gain_b, gain_post, gain_next, keep=False)
    return y.view(a.shape), normed.view(a.shape)


class NormedLayer:
    """A layer with per-head q / k norms over one set of keys.  The anchored-block draft's projects q from the
    normed input (``wq``) and k, v from ``cat([context, normed input])`` (``wkv``); the multi-token-prediction
    layer's does its own input norm and projects all three from it (``wqkv`` in the place of ``wq``)."""

    __slots__ = ("wq", "wkv", "wo", "wgu", "wd", "eps_in", "eps_q", "eps_k", "eps_post", "eps_next", "hq", "hkv", "d",
                 "scaling", "q_pos", "kv_pos", "inv_freq", "mask", "slots", "grad_slot", "pair")

    def __init__(self, wq, wkv, wo, wgu, wd, eps, heads, scaling, q_pos, kv_pos, inv_freq, mask):
        self.wq, self.wkv, self.wo, self.wgu, self.wd = wq, wkv, wo, wgu, wd
        self.eps_in, self.eps_q, self.eps_k, self.eps_post, self.eps_next = eps
        self.hq, self.hkv, self.d = heads
        self.scaling, self.q_pos, self.kv_pos, self.inv_freq, self.mask = scaling, q_pos, kv_pos, inv_freq, mask
        self.slots, self.grad_slot = (None,) * 4, None

    def constants(self, nq: int, nk: int):
        """See ``LayerStep.constants``; the mask's bounds for ``nq`` query rows and ``nk`` keys come first."""
        lo, hi, block_lo, block_hi, _, _ = A.mask_arguments(self.mask, nq, nk)
        weights = (*(w.w for w in (self.wq, self.wkv, self.wo, self.wd) if w is not None), *_gate_up(self))
        return (lo, hi, block_lo, block_hi, self.q_pos, self.kv_pos, self.inv_freq, *weights)

    @staticmethod
    def takes(attention, inv_freq, kernel) -> bool:
        """Whether ``attention`` is one the node's kernels serve (a head size they are built for, the rotary
        embedding over all of it, the attention function ``kernel``)."""
        d = attention.d
        return attention.attn_fn is kernel and d in A.KERNEL_HEAD_DIMS and 2 * inv_freq.numel() == d

    def tokens(self):
        return tuple(w.token for w in (self.wq, self.wkv, self.wo, self.wgu, self.wd) if w is not None)

    def take_slots(self, t: int):
        """See ``LayerStep.take_slots``."""
        self.slots = (self.wq.x_slot(t) if self.wkv is None else None, self.wo.x_slot(t), self.wgu.x_slot(t),
                      self.wd.x_slot(t))


def normed_forward(s: NormedLayer, x, n, context, gain_in, gain_q, gain_k, gain_post, gain_next, keep: bool = True):
    """``(y, normed, saved)`` as in ``step_forward``."""
    x2 = _flat(x)
    nq, h = x2.shape
    dev = x2.device
    slot_in, slot_o, slot_gu, slot_d = s.slots
    rstd_in = None
    if context is not None:
        c2 = _flat(context)
        n2 = _flat(n)
        both = _lib.native().cat_bf16(c2, n2) if c2.is_contiguous() and n2.is_contiguous() else torch.cat((c2, n2))
        n2 = both[c2.shape[0]:]
        q_tok, kv_tok = gemm._project(n2, s.wq), gemm._project(both, s.wkv)
    else:
        rstd_in = torch.empty(nq, device=dev, dtype=torch.float32)
        both = n2 = _rows(slot_in, nq, h, dev)
        _lib.call("spx_rmsnorm_fwd", x2, x2.stride(0), gain_in, n2, h, rstd_in, nq, h, s.eps_in, _lib.stream_ptr(dev))
        q_tok = kv_tok = gemm._project(n2, s.wq)
    q, kv, rq, rk, att, lse = _lib.native().normed_forward(
        q_tok, kv_tok, s.q_pos, s.kv_pos, s.inv_freq, gain_q, gain_k, slot_o, 0 if s.wkv is not None else s.hq * s.d, s.hq,
        s.hkv, s.d, FO.table_scale_of(s.inv_freq), s.scaling, s.eps_q, s.eps_k,
        *A.mask_arguments(s.mask, nq, both.shape[0]))
    y, normed, tail = _tail_forward(s, x2, att, gain_post, gain_next, slot_gu, slot_d, None, keep)
    return y, normed, (x2, rstd_in, both, n2, q_tok, kv_tok, rq, rk, q, kv, att, lse, *tail)


class _NormedLayer(torch.autograd.Function):
    """``(x, norm(x), context, gains, tokens) -> (y, next norm(y))``, or ``(x, None, None, ...)`` with the input
    norm in the node."""

    @staticmethod
    def forward(ctx, s: NormedLayer, x, n, context, gain_in, gain_q, gain_k, gain_post, gain_next, *_tokens):
        y, normed, saved = normed_forward(s, x, n, context, gain_in, gain_q, gain_k, gain_post, gain_next)
        (_, _, both, n2, _, _, _, _, _, _, att, _, _, _, z, _, act, _) = saved
        ctx.taken = (s.wq.take(n2), s.wkv.take(both) if s.wkv is not None else -1, s.wo.take(att), s.wgu.take(z),
                     s.wd.take(act))
        gains = (gain_in, gain_q, gain_k, gain_post, gain_next)
        ctx.gain_grads = tuple(getattr(g, "spx_gain_grads", None) for g in gains)
        ctx.step, ctx.shape, ctx.n_inputs = s, x.shape, 9 + len(_tokens)
        ctx.context_shape = context.shape if context is not None else None
        ctx.save_for_backward(*saved, *gains, *s.constants(n2.shape[0], both.shape[0]))
        ctx.set_materialize_grads(False)
        return y.view(x.shape), normed.view(x.shape)

    @staticmethod
    def backward(ctx, dy, dn):
        s = ctx.step
        if dy is None and dn is None:
            return (None,) * ctx.n_inputs
        (x2, rstd_in, both, n2, q_tok, kv_tok, rq, rk, q, kv, att, lse, mid, stats, z, gu, act, y, gain_in, gain_q, gain_k,
         gain_post, gain_next, *bounds, q_pos, kv_pos, inv_freq) = ctx.saved_tensors[:30]
        tail = (mid, stats, z, gu, act, y)
        needs = ctx.needs_input_grad
        nq, h = n2.shape
        nk = both.shape[0]
        dev = n2.device
        grads_in, grads_q, grads_k, grads_post, grads_next = ctx.gain_grads
        da, datt, d_post, d_next, tok_o, tok_gu, tok_d = _tail_backward(
            s, dy, dn, att, tail, gain_post, gain_next, grads_post, grads_next, needs[7:9], ctx.taken[2:])
        sum_q, sum_k = _GainSum(grads_q, needs[5], nq * s.hq, s.d, dev), _GainSum(grads_k, needs[6], nk * s.hkv, s.d, dev)
        two = s.wkv is not None
        dq_tok, dkv_tok = _lib.native().normed_backward(
            q_tok, kv_tok, q, kv, rq, rk, att, datt, lse, q_pos, kv_pos, inv_freq, gain_q, gain_k,
            s.wq.dy_slot(ctx.taken[0], nq), s.wkv.dy_slot(ctx.taken[1], nk) if two else None, sum_q.scratch, sum_q.acc,
            sum_k.scratch, sum_k.acc, 0 if two else s.hq * s.d, FO.table_scale_of(s.inv_freq), s.scaling, *bounds,
            *A.mask_arguments(s.mask, nq, nk)[4:])
        d_gq, d_gk = sum_q.result(), sum_k.result()
        d_n = gemm._project_back(dq_tok, s.wq)
        tokens = [s.wq.defer(ctx.taken[0], dq_tok, n2)]
        d_context = d_in = None
        if two:
            d_both = gemm._project_back(dkv_tok, s.wkv)
            tokens.append(s.wkv.defer(ctx.taken[1], dkv_tok, both))
            d_n += d_both[nk - nq:]
            d_context = d_both[:nk - nq].view(ctx.context_shape) if needs[3] else None
            dx, d_n = da.view(ctx.shape), d_n.view(ctx.shape)
        else:
            dx = _grad_rows(s.grad_slot, nq, h, dev)
            d_in = FO._norm_backward(grads_in, needs[4], x2, gain_in, d_n, da, rstd_in, dx, nq, h)
            dx, d_n = dx.view(ctx.shape), None
        return (None, dx, d_n, d_context, d_in, d_gq, d_gk, d_post, d_next, *tokens, tok_o, tok_gu, tok_d)


def _grad_rows(grad_slot, rows: int, cols: int, device):
    """Where the gradient of a ``gemm.linear_staged`` result goes: the place its weight gradient reads it from,
    if that has one."""
    if grad_slot is not None and grad_slot[2] == rows:
        out = grad_slot[0].dy_slot(grad_slot[1], rows)
        if out.shape == (rows, cols) and out.is_contiguous():
            return out
    return torch.empty(rows, cols, device=device, dtype=torch.bfloat16)


def run_normed(s: NormedLayer, x, n, context, gain_in, gain_q, gain_k, gain_post, gain_next):
    """``(y, normed)``: the layer's output and the next norm of it."""
    if torch.is_grad_enabled():
        s.grad_slot = getattr(x, "spx_grad_slot", None)
        return _NormedLayer.apply(s, x, n, context, gain_in, gain_q, gain_k, gain_post, gain_next, *s.tokens())
    y, normed, _ = normed_forward(s, x, n, context, gain_in, gain_q, gain_k, gain_post, gain_next, keep=False)
    return y.view(x.shape), normed.view(x.shape)
