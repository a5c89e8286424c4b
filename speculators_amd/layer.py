"""One TTT step of a draft decoder layer as ONE autograd node.

The layer (models/eagle3/model_definitions.py:14-110) is nine launches forward and thirteen backward; as
eight nodes of their own they cost more host time (a node's forward and backward 20 us, and the views,
slot look-ups and gradient checks between them) than the kernels take up to a thousand tokens: at 512
tokens of the 1B shape a step of forward and backward was 0.61 ms of host time, 0.33 ms as one node.
Nothing is computed differently: the same kernels in the same order, on the same buffers
(``weights.Staged`` slots, the layer's K / V cache).
"""

from __future__ import annotations

import torch

from . import _lib
from . import attention as A
from . import fused_ops as FO
from . import gemm


class LayerStep:
    """What a step needs besides its differentiable inputs."""

    __slots__ = ("first", "wqkv", "wo", "wgu", "wd", "eps_in", "eps_post", "eps_next", "hq", "hkv", "d", "scaling",
                 "offset", "positions", "inv_freq", "cache", "mask", "slots")

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


def _rows(t, rows, cols, device):
    return t if t is not None else torch.empty(rows, cols, device=device, dtype=torch.bfloat16)


def _flat(x):
    x2 = x.reshape(-1, x.shape[-1])
    return x2 if x2.stride(1) == 1 else x2.contiguous()


def step_forward(s: LayerStep, a, b, gain_a, gain_b, gain_post, gain_next):
    """``(y, normed, saved)``: the layer's output ``[T, H]``, the next norm of it, and what the backward reads."""
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
    hq, hkv, d = s.hq, s.hkv, s.d
    qkv = gemm._project(xin, s.wqkv)
    scale = FO.table_scale_of(s.inv_freq)
    q, _, _ = gemm._qkv_heads(qkv, s.positions, s.inv_freq, hq, hkv, d, s.offset, scale, s.cache.window(s.offset))
    n = (s.offset + 1) * t
    k, v = s.cache.k[:, :, :n], s.cache.v[:, :, :n]
    att = _rows(slot_o, t, hq * d, dev)
    lse = A.ttt_forward_into(q, k, v, s.mask, s.scaling, att)
    o = gemm._project(att, s.wo)
    stats = torch.empty(2, t, device=dev, dtype=torch.float32)
    mid = torch.empty(t, h, device=dev, dtype=torch.bfloat16)
    z = _rows(slot_gu, t, h, dev)
    _lib.call("spx_add_rmsnorm_fwd", residual, residual.stride(0), o, h, mid, h, gain_post, z, h, stats, t, h,
              s.eps_post, st)
    gu = gemm._project(z, s.wgu)
    f = gu.shape[1] // 2
    act = _rows(slot_d, t, f, dev)
    base = gu.data_ptr()
    _lib.call("spx_swiglu_rows_fwd", base, 2 * f, base + 2 * f, 2 * f, act, f, t, f, st)
    m = gemm._project(act, s.wd)
    y = torch.empty(t, h, device=dev, dtype=torch.bfloat16)
    normed = _rows(slot_next, t, h, dev)
    _lib.call("spx_add_rmsnorm_fwd", mid, h, m, h, y, h, gain_next, normed, h, stats[1], t, h, s.eps_next, st)
    return y, normed, (a2, b2, rstd_in, xin, q, att, lse, mid, stats, z, gu, act, y)


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
        ctx.save_for_backward(*saved, gain_a, gain_b, gain_post, gain_next)
        ctx.set_materialize_grads(False)
        return y.view(shape), normed.view(shape)

    @staticmethod
    def backward(ctx, dy, dn):
        if dy is None and dn is None:
            return (None,) * 11
        (a2, b2, rstd_in, xin, q, att, lse, mid, stats, z, gu, act, y,
         gain_a, gain_b, gain_post, gain_next) = ctx.saved_tensors
        s = ctx.step
        needs = ctx.needs_input_grad
        t, h = y.shape
        f = act.shape[1]
        dev = y.device
        st = _lib.stream_ptr(dev)
        slot_qkv, slot_o, slot_gu, slot_d = ctx.taken
        grads_a, grads_b, grads_post, grads_next = ctx.gain_grads
        if dy is not None:
            dy = _flat(dy).to(torch.bfloat16)
        dm = _rows(s.wd.dy_slot(slot_d, t), t, h, dev)
        d_next = None
        if dn is not None:
            d_next = FO._norm_backward(grads_next, needs[6], y, gain_next, _flat(dn).to(torch.bfloat16), dy, stats[1],
                                       dm, t, h)
        else:
            dm.copy_(dy)
        dact = gemm._project_back(dm, s.wd)
        tok_d = s.wd.defer(slot_d, dm, act)
        dgu = _rows(s.wgu.dy_slot(slot_gu, t), t, 2 * f, dev)
        base, dbase = gu.data_ptr(), dgu.data_ptr()
        _lib.call("spx_swiglu_rows_bwd", base, 2 * f, base + 2 * f, 2 * f, dact, f, dbase, 2 * f, dbase + 2 * f, 2 * f,
                  t, f, st)
        dz = gemm._project_back(dgu, s.wgu)
        tok_gu = s.wgu.defer(slot_gu, dgu, z)
        da = _rows(s.wo.dy_slot(slot_o, t), t, h, dev)
        d_post = FO._norm_backward(grads_post, needs[5], mid, gain_post, dz, dm, stats[0], da, t, h)
        datt = gemm._project_back(da, s.wo)
        tok_o = s.wo.defer(slot_o, da, att)
        step_no = s.offset + 1
        k, v = s.cache.k[:, :, :step_no * t], s.cache.v[:, :, :step_no * t]
        dq, dk, dv = A.ttt_backward_shared(s.cache.grads, q, k, v, att, datt, lse, s.mask, step_no, s.scaling)
        dqkv = _rows(s.wqkv.dy_slot(slot_qkv, t), t, s.wqkv.w.shape[0], dev)
        gemm._qkv_tokens(dqkv, (dq, dk, dv), s.positions, s.inv_freq, s.hq, s.hkv, s.d, s.offset,
                         FO.table_scale_of(s.inv_freq))
        dxin = gemm._project_back(dqkv, s.wqkv)
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
    y, normed, _ = step_forward(s, a, b, gain_a, gain_b, gain_post, gain_next)
    return y.view(a.shape), normed.view(a.shape)
