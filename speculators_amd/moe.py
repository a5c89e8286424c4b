"""Sparse MoE MLP of the hybrid MTP flavours on the HIP path.

The layer is the library's ``Qwen3NextSparseMoeBlock`` (``modeling_qwen3_next.py``; the
``qwen3_5_moe`` block is the same with the renormalisation always on), which the reference
reaches by wrapping ``Qwen3NextDecoderLayer`` / ``Qwen3_5MoeDecoderLayer``
(models/mtp/model_definitions.py:159-205).  The library walks over the experts that were hit and
gathers each one's tokens; here the ``(token, slot)`` pairs are sorted by expert once per call and
every product -- gate/up, down, their input gradients and their weight gradients -- is ONE grouped
launch over all experts (``spx_gemm_bf16_nt_grouped`` / ``_nn_grouped`` on the weights as they lie /
``spx_gemm_bf16_tn_grouped``), with the group boundaries kept on the device: the host never learns
how many tokens an expert received.
"""

from __future__ import annotations

import torch
import torch.nn.functional as F

from . import _lib
from .weights import Staged


def gemm_nt_grouped(a: torch.Tensor, b: torch.Tensor, offsets: torch.Tensor,
                    out: torch.Tensor | None = None) -> torch.Tensor:
    """``out[r] = a[r] @ b[e].T`` for the rows ``offsets[e] <= r < offsets[e + 1]``: ``a [rows, K]``
    sorted by group, ``b [groups, N, K]``, ``offsets`` int32 ``[groups + 1]`` on the device."""
    if a.dtype != torch.bfloat16 or b.dtype != torch.bfloat16:
        raise _lib.SpxError("gemm_nt_grouped takes bf16 operands")
    if a.dim() != 2 or b.dim() != 3 or a.shape[1] != b.shape[2] or not b.is_contiguous():
        raise ValueError(f"shape mismatch: a {tuple(a.shape)} b {tuple(b.shape)} (b contiguous)")
    groups, n, k = b.shape
    if offsets.dtype != torch.int32 or offsets.numel() != groups + 1 or offsets.device != a.device:
        raise ValueError("offsets must be an int32 [groups + 1] tensor on the operands' device")
    if a.stride(1) != 1:
        a = a.contiguous()
    rows = a.shape[0]
    if out is None:
        out = torch.empty(rows, n, device=a.device, dtype=torch.bfloat16)
    nbytes = int(_lib.native().spx_gemm_grouped_workspace_bytes(rows, groups))
    ws = torch.empty(nbytes // 4, device=a.device, dtype=torch.int32)
    _lib.call("spx_gemm_bf16_nt_grouped", a, a.stride(0), b, b.stride(1), b.stride(0),
              out, out.stride(0), rows, n, k, offsets, groups, ws, nbytes,
              _lib.stream_ptr(a.device))
    return out


def gemm_nn_grouped(a: torch.Tensor, b: torch.Tensor, offsets: torch.Tensor,
                    out: torch.Tensor | None = None) -> torch.Tensor:
    """``out[r] = a[r] @ b[e]`` for the rows ``offsets[e] <= r < offsets[e + 1]``: ``a [rows, K]``
    sorted by group, ``b [groups, K, N]`` -- the input gradient of ``gemm_nt_grouped`` against the same
    weight stack as it lies."""
    if a.dtype != torch.bfloat16 or b.dtype != torch.bfloat16:
        raise _lib.SpxError("gemm_nn_grouped takes bf16 operands")
    if a.dim() != 2 or b.dim() != 3 or a.shape[1] != b.shape[1] or not b.is_contiguous():
        raise ValueError(f"shape mismatch: a {tuple(a.shape)} b {tuple(b.shape)} (b contiguous)")
    groups, k, n = b.shape
    if offsets.dtype != torch.int32 or offsets.numel() != groups + 1 or offsets.device != a.device:
        raise ValueError("offsets must be an int32 [groups + 1] tensor on the operands' device")
    if a.stride(1) != 1:
        a = a.contiguous()
    rows = a.shape[0]
    if out is None:
        out = torch.empty(rows, n, device=a.device, dtype=torch.bfloat16)
    nbytes = int(_lib.native().spx_gemm_grouped_workspace_bytes(rows, groups))
    ws = torch.empty(nbytes // 4, device=a.device, dtype=torch.int32)
    _lib.call("spx_gemm_bf16_nn_grouped", a, a.stride(0), b, b.stride(1), b.stride(0),
              out, out.stride(0), rows, n, k, offsets, groups, ws, nbytes,
              _lib.stream_ptr(a.device))
    return out


def gemm_tn_grouped(a: torch.Tensor, b: torch.Tensor, offsets: torch.Tensor, out: torch.Tensor,
                    accumulate: bool = False) -> torch.Tensor:
    """``out[e] (+)= a[rows of e].T @ b[rows of e]``: ``a [rows, M]``, ``b [rows, N]`` sorted by
    group, ``out [groups, M, N]`` bf16 or fp32 -- the weight gradients of all experts."""
    if a.dtype != torch.bfloat16 or b.dtype != torch.bfloat16:
        raise _lib.SpxError("gemm_tn_grouped takes bf16 operands")
    if a.dim() != 2 or b.dim() != 2 or a.shape[0] != b.shape[0]:
        raise ValueError(f"shape mismatch: a {tuple(a.shape)} b {tuple(b.shape)}")
    groups = offsets.numel() - 1
    m, n = a.shape[1], b.shape[1]
    if out.shape != (groups, m, n) or not out.is_contiguous() or out.dtype not in (torch.bfloat16, torch.float32):
        raise ValueError(f"out must be a contiguous bf16 or fp32 [{groups}, {m}, {n}] tensor")
    if offsets.dtype != torch.int32 or offsets.device != a.device:
        raise ValueError("offsets must be an int32 tensor on the operands' device")
    if a.stride(1) != 1:
        a = a.contiguous()
    if b.stride(1) != 1:
        b = b.contiguous()
    _lib.call("spx_gemm_bf16_tn_grouped", a, a.stride(0), b, b.stride(0), out,
              out.stride(1), out.stride(0), m, n, a.shape[0], offsets, groups,
              int(out.dtype == torch.float32), int(accumulate), _lib.stream_ptr(a.device))
    return out


def gemm_tn_grouped_multi(a: torch.Tensor, b: torch.Tensor, offsets: torch.Tensor, out: torch.Tensor,
                          accumulate: bool = False) -> torch.Tensor:
    """The grouped weight gradient over several uses at once: ``a [S * rows, M]`` and
    ``b [S * rows, N]`` are S segments of ``rows`` sorted rows each, ``offsets [S, groups + 1]``
    holds every segment's group boundaries (a row of zeros: that segment has nothing), and
    ``out[e] (+)= sum_s a[rows of e in s].T @ b[rows of e in s]``."""
    segments, g1 = offsets.shape
    rows = a.shape[0] // segments
    m, n = a.shape[1], b.shape[1]
    if (a.dtype != torch.bfloat16 or b.dtype != torch.bfloat16 or a.shape[0] != segments * rows
            or b.shape[0] != a.shape[0] or not a.is_contiguous() or not b.is_contiguous()):
        raise ValueError("a and b must be contiguous bf16 stacks of equally long segments")
    if out.shape != (g1 - 1, m, n) or not out.is_contiguous() or out.dtype not in (torch.bfloat16, torch.float32):
        raise ValueError(f"out must be a contiguous bf16 or fp32 [{g1 - 1}, {m}, {n}] tensor")
    if offsets.dtype != torch.int32 or not offsets.is_contiguous() or offsets.device != a.device:
        raise ValueError("offsets must be a contiguous int32 tensor on the operands' device")
    _lib.call("spx_gemm_bf16_tn_grouped_multi", a, m, b, n, out, n, m * n, m, n,
              rows, segments, offsets, g1 - 1, int(out.dtype == torch.float32), int(accumulate),
              _lib.stream_ptr(a.device))
    return out


def gather_rows(x2: torch.Tensor, src_row: torch.Tensor, scale: torch.Tensor | None = None,
                out: torch.Tensor | None = None) -> torch.Tensor:
    """``out[p] = scale[p] * x2[src_row[p]]`` (bf16 rows, ``src_row`` int32, ``scale`` fp32)."""
    rows, h = src_row.numel(), x2.shape[1]
    if out is None:
        out = torch.empty(rows, h, device=x2.device, dtype=torch.bfloat16)
    _lib.call("spx_moe_gather_rows", x2, x2.stride(0), x2.shape[0], src_row,
              scale, out, h, rows, h, _lib.stream_ptr(x2.device))
    return out


def combine_rows(sorted_rows: torch.Tensor, pos: torch.Tensor, weight: torch.Tensor | None) -> torch.Tensor:
    """``out[t] = sum_j weight[t, j] * sorted_rows[pos[t, j]]`` (``pos`` int32 ``[T, k]``)."""
    tokens, k = pos.shape
    h = sorted_rows.shape[1]
    out = torch.empty(tokens, h, device=sorted_rows.device, dtype=torch.bfloat16)
    _lib.call("spx_moe_combine_rows", sorted_rows, sorted_rows.stride(0), sorted_rows.shape[0],
              pos, weight, out, h, tokens, k, h,
              _lib.stream_ptr(sorted_rows.device))
    return out


def pair_dot(a: torch.Tensor, sorted_rows: torch.Tensor, pos: torch.Tensor) -> torch.Tensor:
    """``out[t, j] = <a[t], sorted_rows[pos[t, j]]>`` in fp32."""
    tokens, k = pos.shape
    out = torch.empty(tokens, k, device=a.device, dtype=torch.float32)
    _lib.call("spx_moe_pair_dot", a, a.stride(0), sorted_rows, sorted_rows.stride(0),
              sorted_rows.shape[0], pos, out, tokens, k, a.shape[1],
              _lib.stream_ptr(a.device))
    return out


def route(logits: torch.Tensor, top_k: int, renormalise: bool):
    """``Qwen3NextTopKRouter.forward`` after the router product: soft-max over all experts in
    fp32, the ``top_k`` largest, optionally renormalised, cast to the logits' dtype.
    -> (scores ``[T, k]``, expert ids ``[T, k]``)."""
    probs = F.softmax(logits, dtype=torch.float, dim=-1)
    top, idx = torch.topk(probs, top_k, dim=-1)
    if renormalise:
        top = top / top.sum(dim=-1, keepdim=True)
    return top.to(logits.dtype), idx


SORT_MAX_EXPERTS = 2048  # of spx_moe_sort_pairs


def sort_pairs(idx: torch.Tensor, num_experts: int):
    """The ``(token, slot)`` pairs of ``idx [T, k]`` sorted by expert (stable: token order inside an
    expert).  -> ``order`` (pair of every sorted row, int64), ``src_row`` (its token, int32),
    ``pos`` (sorted row of every pair, int32 ``[T, k]``), ``offsets`` (int32 ``[E + 1]``).  All on
    the device; nothing is read back."""
    t, k = idx.shape
    dev = idx.device
    pairs = t * k
    idx = idx.to(torch.int64).contiguous()
    order = torch.empty(pairs, device=dev, dtype=torch.int64)
    ints = torch.empty(2 * pairs + num_experts + 1, device=dev, dtype=torch.int32)
    src_row, pos, offsets = ints[:pairs], ints[pairs:2 * pairs], ints[2 * pairs:]
    if idx.is_cuda and num_experts <= SORT_MAX_EXPERTS and pairs:
        nbytes = int(_lib.native().spx_moe_sort_workspace_bytes(pairs, num_experts))
        ws = torch.empty(nbytes // 4, device=dev, dtype=torch.int32)
        _lib.call("spx_moe_sort_pairs", idx, t, k, num_experts, order, src_row,
                  pos, offsets, ws, nbytes, _lib.stream_ptr(dev))
        return order, src_row, pos.view(t, k), offsets
    # host tensors, and more experts than the kernel's counters hold in LDS
    flat = idx.reshape(-1)
    order = torch.argsort(flat, stable=True)
    counts = torch.zeros(num_experts, device=dev, dtype=torch.int32)
    counts.index_add_(0, flat, torch.ones_like(flat, dtype=torch.int32))
    offsets[0] = 0
    offsets[1:] = counts.cumsum(0)
    src_row.copy_(order // k)
    pos[order] = torch.arange(pairs, device=dev, dtype=torch.int32)
    return order, src_row, pos.view(t, k), offsets


PICK_ROWS = 256  # rows a group on average that the picked products take
PICK_BYTES = 0x7ffffff0


class _Picked:
    """The expert products on tokens' rows as they lie: row r of an operand is row ``src_row[r]`` of the tokens'
    matrix (a few MB that the caches hold), looked up by the product's own loads.  The four products of a forward and
    backward share one table of tile rows.

    On copies in sorted order / picked, us: 4096 tokens, top 10 of 512 experts of 512 (a copy: 48), forward 414 / 399,
    input gradient 238 / 223, weight gradients 612 + 321 / 520 + 291; 1500, 8 of 128 (17): 141 / 134, 79 / 76, 163 + 85
    / 127 + 69; 2048, 8 of 64 of 768, 256 rows each (21): 141 / 140, 74 / 66, 181 + 98 / 168 + 91; 12000, 10 of 512, 234
    rows each (141): 672 / 637, 358 / 343, 946 + 465 / 965 + 471."""

    def __init__(self, src_row, off):
        self.src_row, self.off, self.table = src_row, off, None

    @staticmethod
    def takes(x2, rows: int, experts: int) -> bool:
        """Whether ``x2``'s rows are picked (else they are copied into sorted order first, by a launch with rules of its own
        for strides and alignment): few rows an expert (above 256 the products take tall tiles, are bound by their
        arithmetic and have no picked form) and a matrix that 32-bit offsets reach once it is contiguous."""
        return (0 < rows <= PICK_ROWS * experts and x2.shape[0] * x2.shape[1] * 2 < PICK_BYTES
                and x2.stride(0) >= x2.shape[1] and x2.stride(0) % 8 == 0 and x2.data_ptr() % 16 == 0)

    def rows_of(self, form: int, a, b, picked: bool):
        """``a[src_row]`` (``picked``) or ``a`` times every expert's ``b.T`` (form 0) or ``b`` (form 1)."""
        groups, n, k = b.shape if form == 0 else (b.shape[0], b.shape[2], b.shape[1])
        rows = self.src_row.numel()
        if (b.dtype != torch.bfloat16 or a.shape[1] != k or not b.is_contiguous() or self.off.numel() != groups + 1
                or (not picked and a.shape[0] != rows)):
            raise ValueError(f"shape mismatch: a {tuple(a.shape)} b {tuple(b.shape)} (b bf16, contiguous)")
        native = _lib.native()
        nbytes = int(native.spx_gemm_grouped_workspace_bytes(rows, groups))
        ready = self.table is not None
        if not ready:
            self.table = torch.empty(nbytes // 4, device=a.device, dtype=torch.int32)
        out = torch.empty(rows, n, device=a.device, dtype=torch.bfloat16)
        _lib.call("spx_gemm_bf16_grouped_picked", form, a, a.stride(0), self.src_row if picked else None, a.shape[0], b,
                  b.stride(1), b.stride(0), out, n, rows, n, k, self.off, groups, self.table, nbytes, int(ready),
                  _lib.stream_ptr(a.device))
        return out

    def weight_gradient(self, a, b, operand: int, out, accumulate: bool):
        """``out[e] (+)= a[rows of e].T @ b[rows of e]``, the rows of a (operand 0) or b (1) picked."""
        groups, m, n = out.shape
        src = (a, b)[operand]
        _lib.call("spx_gemm_bf16_tn_grouped_picked", a, a.stride(0), b, b.stride(0), self.src_row, src.shape[0], operand, out, n,
                  m * n, m, n, self.src_row.numel(), self.off, groups, int(out.dtype == torch.float32), int(accumulate),
                  _lib.stream_ptr(a.device))


class _ExpertsMLP(torch.autograd.Function):
    """``Qwen3NextExperts.forward``: ``out[t] = sum_j scores[t, j] * down_e(silu(gate_e x_t) * up_e x_t)``,
    ``e = idx[t, j]``, on expert-sorted rows.  The backward takes the scores at the activation, where a row is
    narrow (``spx_moe_swiglu_bwd``).  The weight gradients of the uses of one forward add
    up in one buffer per weight (``Staged.grad_buffer``: fp32, or bf16 for the only use of bf16
    parameters), which the staging node hands to
    autograd once."""

    @staticmethod
    def forward(ctx, x2, scores, idx, _tok_gu, _tok_dn, st_gu: Staged, st_dn: Staged):
        if x2.dtype != torch.bfloat16:
            raise _lib.SpxError("the HIP layer kernels take bf16 tensors")
        w_gu, w_dn = st_gu.w, st_dn.w  # [E, 2I, H], [E, H, I]
        st_gu.applied += 1
        st_dn.applied += 1
        e, i2, _ = w_gu.shape
        inter = i2 // 2
        order, src_row, pos, off = sort_pairs(idx, e)
        rows = src_row.numel()
        st = _lib.stream_ptr(x2.device)
        picked = None
        if x2.stride(1) != 1:
            x2 = x2.contiguous()
        if _Picked.takes(x2, rows, e):
            # (the products' 32-bit offsets span the rows as they lie: of a column slice of a wide buffer, a copy is picked;
            # and one where the backward reads the tokens, which the caller may write to by then: 4096 x 2048 14 us of 2296,
            # 18 on torch's clone)
            picked, xs = _Picked(src_row, off), x2.contiguous()
            if ctx.needs_input_grad[3] and xs.data_ptr() == x2.data_ptr():
                xs = _lib.native().cat_bf16(xs)
            hid = picked.rows_of(0, xs, w_gu, True)
            if not ctx.needs_input_grad[3]:
                xs = None
        else:
            xs = gather_rows(x2, src_row)
            hid = gemm_nt_grouped(xs, w_gu, off)
        act = torch.empty(rows, inter, device=x2.device, dtype=torch.bfloat16)
        up = hid[:, inter:]
        _lib.call("spx_swiglu_rows_fwd", hid, i2, up, i2, act, inter, rows,
                  inter, st)
        wts = scores.float().contiguous()
        ys = gemm_nt_grouped(act, w_dn, off) if picked is None else picked.rows_of(0, act, w_dn, False)
        out = combine_rows(ys, pos, wts)
        ctx.save_for_backward(xs, hid, pos, src_row, off, order, wts)
        ctx.picked = picked
        ctx.staged = (st_gu, st_dn)
        ctx.score_dtype = scores.dtype
        return out

    @staticmethod
    def backward(ctx, dout):
        xs, hid, pos, src_row, off, order, wts = ctx.saved_tensors
        st_gu, st_dn = ctx.staged
        rows, i2 = hid.shape
        inter = i2 // 2
        dout = dout.to(torch.bfloat16).contiguous()
        st = _lib.stream_ptr(dout.device)
        want_gu, want_dn = ctx.needs_input_grad[3], ctx.needs_input_grad[4]
        picked = ctx.picked
        if picked is not None:
            dys = dout
            dact = picked.rows_of(1, dout, st_dn.w, True)
        else:
            dys = gather_rows(dout, src_row)
            dact = gemm_nn_grouped(dys, st_dn.w, off)
        dh = torch.empty(rows, i2, device=dout.device, dtype=torch.bfloat16)
        act = torch.empty(rows, inter, device=dout.device, dtype=torch.bfloat16) if want_dn else None
        dscores = None
        if ctx.needs_input_grad[1]:
            dscores = torch.empty(wts.shape, device=dout.device, dtype=ctx.score_dtype if ctx.score_dtype == torch.bfloat16
                                  else torch.float32)
        _lib.call("spx_moe_swiglu_bwd", hid, i2, order, wts, dact, inter, dh, i2, act, inter, dscores,
                  int(dscores is not None and dscores.dtype == torch.float32), rows, inter, st)
        # The weight gradients before the input gradient, the narrow operand first: act and dh have just been written (126 MB
        # for 40960 rows) and are read out of the memory-side cache, which the input gradient's pass over the weights (2.1 GB)
        # would leave empty.  4096 tokens, top 10 of 512 experts: 621 + 322 -> 537 + 276 us, the pass 2458 -> 2310.
        marks = {}
        for need, staged, dy2, x2, tokens in ((want_dn, st_dn, dys, act, 0), (want_gu, st_gu, dh, xs, 1)):
            if not need:
                continue
            buf, holds = staged.grad_buffer()
            if picked is not None:
                picked.weight_gradient(dy2, x2, tokens, buf, holds)
            else:
                gemm_tn_grouped(dy2, x2, off, buf, accumulate=holds)
            marks[staged] = staged.mark()
        dx = None
        if ctx.needs_input_grad[0]:
            dxs = gemm_nn_grouped(dh, st_gu.w, off) if picked is None else picked.rows_of(1, dh, st_gu.w, False)
            dx = combine_rows(dxs, pos, None)
        return dx, None if dscores is None else dscores.to(ctx.score_dtype), None, marks.get(st_gu), marks.get(st_dn), None, None


def experts_mlp(x2, scores, idx, st_gu: Staged, st_dn: Staged):
    """``[T, H]`` tokens through their ``idx [T, k]`` experts, weighted by ``scores [T, k]``."""
    return _ExpertsMLP.apply(x2, scores, idx, st_gu.token, st_dn.token, st_gu, st_dn)
