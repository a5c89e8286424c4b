"""Loss-function registry backed by the HIP fused vocabulary loss.

Mirror of the reference's loss plug-in (``speculators/losses/utils.py``): a
``LossConfig`` is ``{name: (fn(logits, targets) -> [B, T] float32, weight)}``
(losses/utils.py:12-14) and ``resolve_loss_config(spec, implementation)``
(losses/utils.py:184-230) turns ``"kl_div"`` or a JSON dict of weights into
one.  The implementation name registered here is ``"hip"``; its functions are
differentiable with respect to ``logits`` only, like the reference's fused
losses (losses/fused.py:238-291).
"""

from __future__ import annotations

import json
from collections.abc import Callable
from dataclasses import dataclass

import torch

from . import _lib

LossConfig = dict[str, tuple[Callable[[torch.Tensor, torch.Tensor], torch.Tensor], float]]

OP_KL, OP_RKL, OP_JSD, OP_CE, OP_TV = 0, 1, 2, 3, 4
_NLA_EPS = 1e-5  # losses/fused.py:294


def _rows_2d(t: torch.Tensor) -> torch.Tensor:
    """[B, T, V] -> [B*T, V] view with unit inner stride (copies only if the
    vocabulary axis itself is strided or the rows are not equally spaced)."""
    v = t.shape[-1]
    if t.stride(-1) != 1:
        t = t.contiguous()
    try:
        return t.view(-1, v)
    except RuntimeError:
        return t.reshape(-1, v)


@dataclass
class StepPass:
    """What one TTT step adds to the row pass of the loss kernel (``spx_vocab_loss_step_fwd``).

    ``d2t`` (int64 ``[Vd]``): the targets are FULL-vocabulary verifier rows and target element i
    is read at column ``i + d2t[i]`` while streaming; the draft-vocabulary rows come back in
    ``gathered`` (``[rows, Vd]``) for the later steps and the backward.
    ``counts`` (int32 ``[3]``, zeroed; None in front of ``_loss_step``, which has its own): the acceptance chain is
    done row by row in the same pass (``mask`` / ``prev`` are the step's 1-D views, ``prev`` is updated in place).
    ``grad_in_pass``: a promise of the caller that the reduction behind the row losses gives a row
    whose ``mask`` entry is zero the weight zero (the masked mean of ``compute_metrics`` does).  The
    head + loss node may then leave the gradient of the logits behind in the same row pass
    (``spx_vocab_loss_step_fwd_grad``) instead of reading both rows again in its backward; masked
    rows get no gradient whatever arrives for them."""

    d2t: torch.Tensor | None = None
    gathered: torch.Tensor | None = None
    mask: torch.Tensor | None = None
    prev: torch.Tensor | None = None
    counts: torch.Tensor | None = None
    grad_in_pass: bool = False


def fused_loss_forward(op: int, logits: torch.Tensor, targets: torch.Tensor, target_stats=None,
                       step: StepPass | None = None):
    """Run the forward kernel.  Returns (loss [R] f32, lse_d, lse_t, extra,
    argmax_draft [R] i32, argmax_target [R] i32, logits2d, targets2d).

    ``target_stats = (lse_target [R] f32, argmax_target [R] i32)`` from an earlier call on
    the same target rows lets kl / ce skip the target row statistics (ce then does not
    read the targets at all).  ``step``: see ``StepPass``; with ``step.d2t`` the returned
    ``targets2d`` are the gathered draft-vocabulary rows."""
    gather = step is not None and step.d2t is not None
    if targets is None:
        # cross-entropy against arg-max targets whose arg-max is known: no target row is read
        if op != OP_CE or target_stats is None or gather:
            raise ValueError("only ce with known target statistics runs without the target rows")
        return _ce_without_targets(logits, target_stats, step)
    if not gather and logits.shape != targets.shape:
        raise ValueError(f"logits {tuple(logits.shape)} and targets {tuple(targets.shape)} differ")
    if gather and logits.shape[:-1] != targets.shape[:-1]:
        raise ValueError(f"logits {tuple(logits.shape)} and full-vocabulary targets "
                         f"{tuple(targets.shape)} differ in their rows")
    if logits.dtype != targets.dtype:
        targets = targets.to(logits.dtype)
    x, y = _rows_2d(logits), _rows_2d(targets)
    rows, vocab = x.shape
    dev = x.device
    if step is not None:
        if gather:
            if target_stats is not None:
                raise ValueError("the gather form computes the target statistics itself")
            if step.d2t.dtype != torch.int64 or step.d2t.numel() != vocab or not step.d2t.is_contiguous():
                raise ValueError("d2t must be a contiguous int64 [draft vocabulary] tensor")
            step.gathered = torch.empty(rows, vocab, device=dev, dtype=x.dtype)
        stats = torch.empty(4, rows, device=dev, dtype=torch.float32)
        arg = torch.empty(2, rows, device=dev, dtype=torch.int32)
        reuse = target_stats is not None and op in (OP_KL, OP_CE)
        lse_t, am_t = stats[2], arg[1]
        if reuse:
            lse_t, am_t = target_stats[0].reshape(-1), target_stats[1].reshape(-1)
        g = step.gathered
        _lib.call(
            "spx_vocab_loss_step_fwd", op, x, x.stride(0), y, y.stride(0),
            step.d2t, y.shape[1] if gather else 0, g if gather else None,
            g.stride(0) if gather else 0, rows, vocab, _lib.dtype_code(x), stats[0],
            stats[1], lse_t, stats[3], arg[0], am_t,
            int(reuse), step.mask, _lib.kind_code(step.mask) if step.mask is not None else 0,
            step.prev, _lib.kind_code(step.prev) if step.prev is not None else 0,
            step.counts, _lib.stream_ptr(dev),
        )
        return stats[0], stats[1], lse_t, stats[3], arg[0], am_t, x, (g if gather else y)
    reuse = target_stats is not None and op in (OP_KL, OP_CE)
    stats = torch.empty(4, rows, device=dev, dtype=torch.float32)
    arg = torch.empty(2, rows, device=dev, dtype=torch.int32)
    lse_t, am_t = stats[2], arg[1]
    if reuse:
        lse_t = target_stats[0].reshape(-1)
        am_t = target_stats[1].reshape(-1)
        if lse_t.numel() != rows or am_t.numel() != rows or lse_t.stride(0) != 1 or am_t.stride(0) != 1:
            raise ValueError("target_stats must be contiguous [rows] tensors")
    _lib.call(
        "spx_fused_vocab_loss_fwd", op, x, x.stride(0), y, y.stride(0),
        rows, vocab, _lib.dtype_code(x), stats[0], stats[1],
        lse_t, stats[3], arg[0], am_t, int(reuse),
        _lib.stream_ptr(dev),
    )
    return stats[0], stats[1], lse_t, stats[3], arg[0], am_t, x, y


def _ce_without_targets(logits, target_stats, step):
    x = _rows_2d(logits)
    rows, vocab = x.shape
    dev = x.device
    stats = torch.empty(4, rows, device=dev, dtype=torch.float32)
    arg = torch.empty(1, rows, device=dev, dtype=torch.int32)
    lse_t, am_t = target_stats[0].reshape(-1), target_stats[1].reshape(-1)
    if lse_t.numel() != rows or am_t.numel() != rows or lse_t.stride(0) != 1 or am_t.stride(0) != 1:
        raise ValueError("target_stats must be contiguous [rows] tensors")
    if step is not None:
        _lib.call(
            "spx_vocab_loss_step_fwd", OP_CE, x, x.stride(0), None, 0, None, 0, None, 0, rows, vocab,
            _lib.dtype_code(x), stats[0], stats[1], lse_t, stats[3],
            arg[0], am_t, 1, step.mask,
            _lib.kind_code(step.mask) if step.mask is not None else 0, step.prev,
            _lib.kind_code(step.prev) if step.prev is not None else 0, step.counts,
            _lib.stream_ptr(dev))
    else:
        _lib.call(
            "spx_fused_vocab_loss_fwd", OP_CE, x, x.stride(0), None, 0, rows, vocab,
            _lib.dtype_code(x), stats[0], stats[1], lse_t, stats[3],
            arg[0], am_t, 1, _lib.stream_ptr(dev))
    return stats[0], stats[1], lse_t, stats[3], arg[0], am_t, x, None


class _FusedLoss(torch.autograd.Function):
    """``(logits, targets, op[, lse_t, am_t]) -> (row_loss [B, T] f32, argmax_draft,
    argmax_target, lse_target)``; the autograd counterpart of ``_FusedLoss`` in
    losses/fused.py:238-291.  Targets get no gradient."""

    @staticmethod
    def forward(ctx, logits, targets, op, known_lse_t=None, known_am_t=None, n_rows=None, step=None):
        known = (known_lse_t, known_am_t) if known_lse_t is not None else None
        # n_rows: only the first n_rows rows of ``logits`` (a [1, T, V] tensor) take part, the
        # rest get a zero gradient.  Doing the cut here instead of slicing outside keeps
        # autograd from materialising a zero-padded copy of the whole gradient.
        ctx.full_shape = logits.shape
        used = logits if n_rows is None else logits[:, :n_rows]
        loss, lse_d, lse_t, extra, am_d, am_t, x, y = fused_loss_forward(op, used, targets, known, step)
        ctx.save_for_backward(x, None if op == OP_CE else y, lse_d, lse_t, extra, am_t)
        ctx.op = op
        lead = used.shape[:-1]
        am_d, am_t, lse_t = am_d.view(lead), am_t.view(lead), lse_t.view(lead)
        ctx.mark_non_differentiable(am_d, am_t, lse_t)
        ctx.set_materialize_grads(False)  # no zero tensors for the outputs that carry no gradient
        return loss.view(lead), am_d, am_t, lse_t

    @staticmethod
    def backward(ctx, grad_rows, _gd, _gt, _gl):
        if grad_rows is None:
            return (None,) * 7
        x, y, lse_d, lse_t, extra, am_t = ctx.saved_tensors
        rows, vocab = x.shape
        full_rows = 1
        for d in ctx.full_shape[:-1]:
            full_rows *= d
        g = grad_rows.reshape(-1).to(torch.float32).contiguous()
        grad = torch.empty(full_rows, vocab, device=x.device, dtype=x.dtype)
        _lib.call(
            "spx_fused_vocab_loss_bwd", ctx.op, x, x.stride(0), y,
            y.stride(0) if y is not None else 0, rows, vocab, _lib.dtype_code(x),
            lse_d, lse_t, extra, am_t, g, None,
            grad, grad.stride(0), _lib.stream_ptr(x.device),
        )
        if full_rows > rows:
            grad[rows:].zero_()
        return grad.view(ctx.full_shape), None, None, None, None, None, None


def _packed_row_map(row_grad: torch.Tensor, labels: torch.Tensor | None = None, ignore_index: int = -100):
    """(row map int32 [rows], live-row count int32 [1]): a row is live when its incoming gradient is
    non-zero (and its label is not the ignored one); live row r goes to slot ``#live rows before
    r``, the others to -1.  One small kernel; the count stays on the device."""
    rows = row_grad.numel()
    out = torch.empty(rows + 1, device=row_grad.device, dtype=torch.int32)
    _lib.call("spx_pack_row_map", row_grad, labels, int(ignore_index), rows,
              out, out[rows:], _lib.stream_ptr(row_grad.device))
    return out[:rows], out[rows:]


def _unpack_rows_scaled(packed: torch.Tensor, row_map: torch.Tensor, row_scale: torch.Tensor, total_rows: int):
    """``_unpack_rows`` with live row r multiplied by ``row_scale[r]`` (fp32) on its way."""
    out = torch.empty(total_rows, packed.shape[1], device=packed.device, dtype=packed.dtype)
    _lib.call("spx_unpack_rows_scaled", packed, packed.stride(0), row_map, row_scale,
              row_map.numel(), total_rows, packed.shape[1], out, out.stride(0),
              _lib.stream_ptr(packed.device))
    return out


# The head + loss node writes the logits gradient in its forward row pass where it can (see StepPass)
HEAD_LOSS_ONE_PASS = True


def _one_pass_ok(op, x, y, step) -> bool:
    if not (HEAD_LOSS_ONE_PASS and step is not None and step.grad_in_pass and step.d2t is None
            and step.mask is not None and op in (OP_KL, OP_CE) and x.dtype == torch.bfloat16):
        return False
    rows, vocab = x.shape
    if rows == 0 or vocab % 8 or vocab > 32768 or x.stride(1) != 1 or x.stride(0) % 8 or x.data_ptr() % 16:
        return False
    if step.mask.numel() != rows or (y is None and op != OP_CE):
        return False
    return y is None or (y.dtype == torch.bfloat16 and y.stride(1) == 1 and y.stride(0) % 8 == 0
                         and y.data_ptr() % 16 == 0)


def _loss_step(op, x, y, known, step, mean=None, total_in=None):
    """The row pass that also writes the unit-weight logits gradient of the unmasked rows, packed to the front, and
    the masked mean behind it.  Returns ``(total, loss, am_d, am_t, lse_t, packed, row_map, count, row_weight, row_of)``
    (``row_of``: the live rows in their order)."""
    rows = x.shape[0]
    lse_t = am_t = None
    if known is not None:
        lse_t, am_t = known[0].reshape(-1), known[1].reshape(-1)
        if lse_t.numel() != rows or am_t.numel() != rows or lse_t.stride(0) != 1 or am_t.stride(0) != 1:
            raise ValueError("target_stats must be contiguous [rows] tensors")
    of_mean = (0.0, 0.0, None) if mean is None else (mean.weight, mean.factor, mean.out)
    return _lib.native().loss_step(
        op, x, y, lse_t, am_t, step.mask, _lib.kind_code(step.mask), step.prev,
        _lib.kind_code(step.prev) if step.prev is not None else 0, step.counts, total_in, *of_mean)


def _loss_forward_with_grad(op, x, y, known, step):
    """``_loss_step`` without the mean: ``(loss, lse_t, am_d, am_t, packed, row_map, count)``."""
    _, loss, am_d, am_t, lse_t, packed, row_map, count, *_ = _loss_step(op, x, y, known, step)
    return loss, lse_t, am_d, am_t, packed, row_map, count


def _unpack_rows(packed: torch.Tensor, row_map: torch.Tensor, total_rows: int):
    """One row per position again: live rows from their packed slot, the others (and the rows past
    the map, up to ``total_rows``) zero.  Slots past the count are never read."""
    out = torch.empty(total_rows, packed.shape[1], device=packed.device, dtype=packed.dtype)
    _lib.call("spx_unpack_rows", packed, packed.stride(0), row_map, row_map.numel(),
              total_rows, packed.shape[1], out, out.stride(0), _lib.stream_ptr(packed.device))
    return out


class _HeadFusedLoss(torch.autograd.Function):
    """A frozen ``lm_head`` and the fused vocabulary loss behind it as ONE autograd node:
    ``(x [T, H], weight [Vd, H], weight_t [H, Vd], targets [n_rows, Vd], op, ...) ->
    (row loss [n_rows], argmax_draft, argmax_target, lse_target, logits [T, Vd])``.

    Rows the loss mask removes (and the rows past ``n_rows``) have an all-zero logits gradient.
    With both steps in one node the backward packs the live rows to the front
    (``spx_fused_vocab_loss_bwd_packed``) and the input-gradient product of the head runs over
    them only (``spx_gemm_bf16_nt_rows``, count read on the device); dead rows of the result are
    exact zeros, as they are when the product runs over all rows.  The logits come back for the
    metrics and the draft tokens and carry no gradient of their own."""

    @staticmethod
    def forward(ctx, x2, weight, weight_t, targets, op, known_lse_t, known_am_t, n_rows, step=None):
        from .gemm import matmul_nt

        logits = matmul_nt(x2, weight)
        known = (known_lse_t, known_am_t) if known_lse_t is not None else None
        ctx.op, ctx.total_rows = op, logits.shape[0]
        loss, lse_d, lse_t, extra, am_d, am_t, x, y = fused_loss_forward(op, logits[:n_rows], targets, known, step)
        ctx.save_for_backward(x, None if op == OP_CE else y, lse_d, lse_t, extra, am_t, weight_t)
        ctx.mark_non_differentiable(am_d, am_t, lse_t, logits)
        ctx.set_materialize_grads(False)  # no [T, Vd] zeros for the logits, which carry no gradient
        return loss, am_d, am_t, lse_t, logits

    @staticmethod
    def backward(ctx, grad_rows, _gd, _gt, _gl, _glogits):
        if grad_rows is None:
            return (None,) * 9
        g = grad_rows.reshape(-1).to(torch.float32).contiguous()
        return (_head_rows_backward(ctx.op, ctx.saved_tensors, g, ctx.total_rows),) + (None,) * 8


def _head_rows_backward(op, saved, g, total_rows):
    """dx of the frozen head behind the row losses whose gradients are ``g`` (f32 ``[rows]``)."""
    from .gemm import matmul_nt

    x, y, lse_d, lse_t, extra, am_t, weight_t = saved
    rows, vocab = x.shape
    row_map, count = _packed_row_map(g)
    packed = torch.empty(rows, vocab, device=x.device, dtype=x.dtype)
    _lib.call(
        "spx_fused_vocab_loss_bwd_packed", op, x, x.stride(0), y,
        y.stride(0) if y is not None else 0, rows, vocab, _lib.dtype_code(x),
        lse_d, lse_t, extra, am_t, g, None,
        row_map, packed, packed.stride(0), _lib.stream_ptr(x.device),
    )
    dx_packed = matmul_nt(packed, weight_t, m_live=count)
    return _unpack_rows(dx_packed, row_map, total_rows)


@dataclass
class MeanTerm:
    """The masked mean behind the row losses of one step (``spx_ttt_step_total``): the step's ``weight``, the
    term's ``factor`` in the loss, and ``out``, which receives the step's scalars (f32 ``[8]``)."""

    mask: torch.Tensor | None
    weight: float
    factor: float
    out: torch.Tensor

    def reduce(self, loss, am_d, am_t, counts, total_in):
        """``(total 0-d, row weights)``: ``total_in`` (or nothing) + the weighted masked mean."""
        n, dev = loss.numel(), loss.device
        row_weight = torch.empty(n, device=dev, dtype=torch.float32)
        total = torch.empty((), device=dev, dtype=torch.float32)
        _lib.call("spx_ttt_step_total", loss, am_d, am_t, self.mask,
                  _lib.kind_code(self.mask) if self.mask is not None else 0, None, 0, n, self.weight, counts,
                  self.factor, total_in, total, self.out, row_weight, _lib.stream_ptr(dev))
        return total, row_weight


@dataclass
class BlockTerm:
    """``MeanTerm`` for a batch of anchored blocks (``spx_block_total``): the weighted masked mean of one term, its
    ``factor`` in the loss, and ``out`` (f32 ``[9 + 2 * block_size]``), which receives the step's scalars.  ``row_weights``:
    weights from the masked row losses (D-PACE) in the place of the exponential decay over the slots."""

    mask: torch.Tensor
    block_size: int
    gamma: float
    from_anchor: bool
    factor: float
    out: torch.Tensor
    row_weights: Callable | None = None

    def reduce(self, loss, am_d, am_t, counts, total_in):
        """As ``MeanTerm.reduce`` (``counts``: none, blocks have no acceptance chain)."""
        n, dev = loss.numel(), loss.device
        pos = None
        if self.row_weights is not None:
            pos = self.row_weights(loss.detach() * self.mask.to(torch.float32)).contiguous()
        row_weight = torch.empty(n, device=dev, dtype=torch.float32)
        total = torch.empty((), device=dev, dtype=torch.float32)
        _lib.call("spx_block_total", loss, am_d, am_t, self.mask, _lib.kind_code(self.mask), pos, float(self.gamma),
                  int(self.from_anchor), n, self.block_size, self.factor, total_in, total, self.out, row_weight,
                  _lib.stream_ptr(dev))
        return total, row_weight


def _unit_rows_backward(saved, g32, factor: float, total_rows: int):
    """dx of the frozen head from the unit-weight logits gradient of the live rows that the row pass left behind: the row
    weights go onto the product's fp32 sums, so that dx is rounded once."""
    from .gemm import rows_graded

    packed, row_map, count, weight_t, row_weight, row_of = saved
    return _unpack_rows(rows_graded(packed, weight_t, count, row_of, row_weight, g32, factor), row_map, total_rows)


class _HeadStepLoss(torch.autograd.Function):
    """``_HeadFusedLoss`` and the masked mean behind it as one node, which also adds the step to the loss so far:
    ``(x, total_in) -> (total, argmax_draft, argmax_target, lse_target, logits)``.

    Where it can (``_one_pass_ok``) the forward reads the rows once for everything: loss, statistics, acceptance
    chain and the unit-weight logits gradient of the unmasked rows, packed to the front; the backward is then the
    input-gradient product of the head, which applies the row weights, and the unpacking of its rows."""

    @staticmethod
    def forward(ctx, x2, total_in, weight, weight_t, targets, op, known, n_rows, step, mean):
        from .gemm import matmul_nt

        logits = matmul_nt(x2, weight)
        ctx.op, ctx.total_rows, ctx.factor = op, logits.shape[0], mean.factor
        xs = logits[:n_rows]
        blocks = isinstance(mean, BlockTerm)
        ctx.one_pass = ((known is not None or targets is not None) and _one_pass_ok(op, xs, targets, step)
                        and (not blocks or xs.shape[1] >= TERMS_MIN_VOCAB))
        if ctx.one_pass:
            total, loss, am_d, am_t, lse_t, packed, row_map, count, row_weight, row_of = _loss_step(
                op, xs, targets, known, step, None if blocks else mean, total_in)
            if blocks:
                total, row_weight = mean.reduce(loss, am_d, am_t, None, total_in)
            ctx.save_for_backward(packed, row_map, count, weight_t, row_weight, row_of)
        else:
            if blocks:
                step = None
            else:
                step.counts = torch.zeros(3, device=x2.device, dtype=torch.int32)
            loss, lse_d, lse_t, extra, am_d, am_t, x, y = fused_loss_forward(op, xs, targets, known, step)
            total, row_weight = mean.reduce(loss, am_d, am_t, None if blocks else step.counts, total_in)
            ctx.save_for_backward(x, None if op == OP_CE else y, lse_d, lse_t, extra, am_t, weight_t, row_weight)
        ctx.mark_non_differentiable(am_d, am_t, lse_t, logits)
        ctx.set_materialize_grads(False)
        return total, am_d, am_t, lse_t, logits

    @staticmethod
    def backward(ctx, g, _gd, _gt, _gl, _glogits):
        if g is None:
            return (None,) * 10
        g32 = g.to(torch.float32)
        if ctx.one_pass:
            dx = _unit_rows_backward(ctx.saved_tensors, g32, ctx.factor, ctx.total_rows)
        else:
            *saved, row_weight = ctx.saved_tensors
            dx = _head_rows_backward(ctx.op, saved, row_weight * (g32 * ctx.factor), ctx.total_rows)
        return (dx, g if ctx.needs_input_grad[1] else None) + (None,) * 8


def head_step_loss(op: int, x, weight, weight_t, targets, target_stats, n_rows: int, step: StepPass, mean: MeanTerm,
                   total_in=None):
    """Head and loss of one step with its masked mean (``mean``) added to ``total_in``: ``(total, argmax_draft,
    argmax_target, lse_target, logits [1, T, Vd])``, the row quantities ``[n_rows]``."""
    y = _check_head(x, weight, targets, n_rows)
    t = x.shape[1]
    total, am_d, am_t, lse_t, logits = _HeadStepLoss.apply(x.reshape(t, x.shape[2]), total_in, weight, weight_t, y, op,
                                                           target_stats, n_rows, step, mean)
    return total, am_d, am_t, lse_t, logits.view(1, t, weight.shape[0])


# From here on a step's terms (and the loss of anchored blocks) share one row pass: a chunk of eight columns for each of the
# row pass's 512 threads.  Three steps of {"ce": 0.1, "tv": 0.9}, forward and backward, head of width 2048, term by term -> one
# pass: 4096 rows of 32000 4.24 -> 2.93 ms, of 8192 1.31 -> 0.97, of 4096 1.06 -> 0.61, of 3072 1.06 -> 0.56, of 2048 1.05 -> 0.45, of
# 1024 1.07 -> 0.42; 512 rows 1.05 -> 0.42 at any width (launches).  So the line is not where the gain ends.  It lies there
# because shorter rows promise more: the two-node form, whose results at short rows the one-node form has to give bit for bit
# (another order of sums in the one pass); at draft vocabularies in earnest (32000) it makes no difference.
TERMS_MIN_VOCAB = 4096


def terms_fit(loss_config, weight, targets, d2t, mask, n_rows: int) -> bool:
    """Whether a step's loss is a sum of terms that the one-read row pass takes (``head_terms_loss``): several terms,
    or one that needs a second walk over the rows, on bf16 rows that fit a workgroup's registers, under a loss mask."""
    if not HEAD_LOSS_ONE_PASS or mask is None or mask.numel() != n_rows or n_rows == 0:
        return False
    ops = [PRIMITIVE_OP.get(name) for name in loss_config]
    if any(op is None or fn is not _HIP_LOSS_FN_MAP[name] for op, (name, (fn, _)) in zip(ops, loss_config.items(), strict=True)):
        return False
    if len(ops) == 1 and ops[0] in (OP_KL, OP_CE):
        return False  # _HeadStepLoss
    vocab = weight.shape[0]
    if vocab % 8 or not TERMS_MIN_VOCAB <= vocab <= 32768 or weight.dtype != torch.bfloat16 or targets.dtype != torch.bfloat16:
        return False
    if d2t is not None:
        return d2t.numel() == vocab
    y = _rows_2d(targets)
    return y.shape[1] == vocab and y.stride(0) % 8 == 0 and y.data_ptr() % 16 == 0


class _HeadTermsLoss(torch.autograd.Function):
    """``_HeadStepLoss`` for a loss of several terms: ``(x, total_in) -> (total, argmax_draft, argmax_target, lse_target,
    logits)``.  The row pass leaves the gradient of their weighted sum behind, so the backward knows no
    terms."""

    @staticmethod
    def forward(ctx, x2, total_in, weight, weight_t, targets, d2t, terms, known, n_rows, step, step_weight, out):
        from .gemm import matmul_nt

        logits = matmul_nt(x2, weight)
        ctx.total_rows = logits.shape[0]
        weights = [0.0] * 5
        for op, w in terms:
            weights[op] = w
        lse_t, am_t = (None, None) if known is None else (known[0].reshape(-1), known[1].reshape(-1))
        total, am_d, am_t, lse_t, packed, row_map, count, row_weight, row_of, rows = _lib.native().loss_terms(
            sum(1 << op for op, _ in terms), *weights, logits[:n_rows], targets, d2t, lse_t, am_t, step.mask,
            _lib.kind_code(step.mask), step.prev, _lib.kind_code(step.prev) if step.prev is not None else 0, total_in,
            step_weight, out)
        ctx.save_for_backward(packed, row_map, count, weight_t, row_weight, row_of)
        if d2t is not None:
            step.gathered = rows
        ctx.mark_non_differentiable(am_d, am_t, lse_t, logits)
        ctx.set_materialize_grads(False)
        return total, am_d, am_t, lse_t, logits

    @staticmethod
    def backward(ctx, g, _gd, _gt, _gl, _glogits):
        if g is None:
            return (None,) * 12
        dx = _unit_rows_backward(ctx.saved_tensors, g.to(torch.float32), 1.0, ctx.total_rows)
        return (dx, g if ctx.needs_input_grad[1] else None) + (None,) * 10


def head_terms_loss(loss_config, x, weight, weight_t, targets, d2t, target_stats, n_rows: int, step: StepPass,
                    step_weight: float, out, total_in=None):
    """One step's whole loss (``terms_fit``) behind the frozen head, added to ``total_in``; ``out`` (f32 ``[18]``) receives
    the scalars of ``spx_ttt_step_terms``.  ``d2t``: ``targets`` are full-vocabulary rows, the gathered ones come back in
    ``step.gathered``.  Returns ``(total, argmax_draft, argmax_target, lse_target, logits [1, T, Vd])``."""
    y = _check_head(x, weight, targets, n_rows)
    if target_stats is not None and any(s.numel() != n_rows or s.stride(-1) != 1 for s in target_stats):
        raise ValueError("target_stats must be contiguous [rows] tensors")
    t = x.shape[1]
    terms = [(PRIMITIVE_OP[name], float(w)) for name, (_, w) in loss_config.items()]
    total, am_d, am_t, lse_t, logits = _HeadTermsLoss.apply(
        x.reshape(t, x.shape[2]), total_in, weight, weight_t, y, d2t, terms, target_stats, n_rows, step, step_weight, out)
    return total, am_d, am_t, lse_t, logits.view(1, t, weight.shape[0])


LOSS_STEPS_MAX = 32            # SPX_LOSS_STEPS_MAX
STEPS_LOGITS_BYTES = 1 << 32   # logits of several steps that are held at a time (at least one step's; fewer where memory is short)


class _HeadStepsLoss(torch.autograd.Function):
    """``_HeadStepLoss`` of all steps of a TTT loop at once: ``(x of every step) -> total``.  A target row meets the draft
    rows of all steps in one workgroup (``spx_loss_steps_pass``), and the backward is ONE input-gradient product over the live
    rows of all steps.  Everything else comes back in ``run``."""

    @staticmethod
    def forward(ctx, run, weight, weight_t, *xs):
        from .gemm import matmul_nt

        t, vocab, steps = run.mask.numel(), weight.shape[0], len(xs)
        dev = weight.device
        native = _lib.native()
        kind = _lib.kind_code(run.mask)
        grad = run.grad
        ints, floats, count, row_slot, slot_row, row_weight = native.loss_steps_begin(run.mask, kind, run.terms, *run.weights)
        run.tokens = torch.empty(steps, t, device=dev, dtype=torch.int64)
        hits = torch.empty(steps, t, device=dev, dtype=torch.uint8)
        packed = torch.empty(steps * t, vocab, device=dev, dtype=torch.bfloat16) if grad else None
        at_once = min(steps, max(1, STEPS_LOGITS_BYTES // (2 * t * vocab)))
        first = 0
        while first < steps:
            logits = None  # (freed before the next are made)
            try:
                logits = [matmul_nt(x.reshape(t, x.shape[-1]), weight) for x in xs[first:first + at_once]]
            except torch.OutOfMemoryError:
                if at_once == 1:
                    raise
                at_once //= 2
                continue
            native.loss_steps_pass(run.op, run.terms, run.masked_first, run.mask, kind, run.targets, run.argmax, ints, floats,
                                   run.tokens, hits, packed, steps, first, *logits)
            if run.logits is not None:
                run.logits += logits
            first += len(logits)
        run.scalars, total = native.loss_steps_end(
            run.terms, run.mask, kind, run.prev, _lib.kind_code(run.prev) if run.prev is not None else 0, ints, floats, hits, steps,
            run.factor)
        if grad:
            ctx.save_for_backward(packed, row_slot, count, weight_t, row_weight, slot_row)
        ctx.factor, ctx.shapes = run.factor, [x.shape for x in xs]
        return total

    @staticmethod
    def backward(ctx, g):
        steps = len(ctx.shapes)
        row_slot = ctx.saved_tensors[1]
        dx = _unit_rows_backward(ctx.saved_tensors, g.to(torch.float32), ctx.factor, row_slot.numel())
        return (None, None, None) + tuple(d.view(shape) for d, shape in zip(dx.chunk(steps), ctx.shapes, strict=True))


@dataclass
class HeadSteps:
    """One loss (``op``: kl or ce) of all steps behind the frozen head, or a sum of several (``terms``: five weights by op, None
    for those that are none): per-step ``weights`` of the masked mean, the one term's ``factor``, 1-D ``mask`` and ``prev`` (advanced in
    place), ``targets`` ``[T, vocab]`` or for ce alone their ``argmax``; ``masked_first``: the first step's masked rows have a loss.
    Filled by ``head_steps_loss``: ``tokens`` int64 ``[steps, T]``, ``scalars`` f32 ``[steps, 8]`` (``spx_ttt_step_total``; of
    several terms ``[steps, 18]``, ``spx_ttt_step_terms``) and, where it is a list before, ``logits``."""

    op: int
    weights: list
    factor: float
    mask: torch.Tensor
    prev: torch.Tensor | None
    targets: torch.Tensor | None
    argmax: torch.Tensor | None
    logits: list | None = None
    terms: tuple | None = None
    masked_first: bool = True
    grad: bool = False
    tokens: torch.Tensor | None = None
    scalars: torch.Tensor | None = None


STEPS_OPS = (OP_KL, OP_CE, OP_TV)  # rkl and jsd do not fit the registers


def steps_fit(loss_config, steps: int, x, weight, mask) -> bool:
    """Whether ``head_steps_loss`` takes the steps: terms of ``STEPS_OPS`` and logits that fit a workgroup's registers, as
    ``_one_pass_ok``, of 4096 columns on as ``TERMS_MIN_VOCAB``.  From two steps on: it has something to share."""
    if not (HEAD_LOSS_ONE_PASS and 2 <= steps <= LOSS_STEPS_MAX and mask is not None):
        return False
    if any(PRIMITIVE_OP.get(name) not in STEPS_OPS or fn is not _HIP_LOSS_FN_MAP[name] for name, (fn, _) in loss_config.items()):
        return False
    t, vocab = mask.numel(), weight.shape[0]
    return (t >= steps and t * steps < 1 << 31 and x.shape[:-1] == (1, t) and x.dtype == weight.dtype == torch.bfloat16
            and vocab % 8 == 0 and TERMS_MIN_VOCAB <= vocab <= 32768)


def steps_rows_fit(rows, t: int, vocab: int) -> bool:
    """Whether ``rows`` can be the target rows of ``head_steps_loss``."""
    return (rows.dtype == torch.bfloat16 and rows.shape == (t, vocab) and rows.stride(1) == 1 and rows.stride(0) % 8 == 0
            and rows.data_ptr() % 16 == 0)


def head_steps_loss(run: HeadSteps, weight, weight_t, xs):
    """The loss of all steps (``steps_fit``) over ``xs``, every step's ``[1, T, H]``, behind the frozen head ``weight``."""
    run.grad = torch.is_grad_enabled() and any(x.requires_grad for x in xs)
    return _HeadStepsLoss.apply(run, weight, weight_t, *xs)


def _check_head(x, weight, targets, n: int):
    if x.dtype != torch.bfloat16 or weight.dtype != torch.bfloat16:
        raise _lib.SpxError("head_fused_rows takes bf16 operands")
    if weight.requires_grad:
        raise ValueError("head_fused_rows is for a frozen head (no weight gradient is produced)")
    if x.dim() != 3 or x.shape[0] != 1:
        raise ValueError("x must be [1, T, H] (the packed batch layout)")
    y = None if targets is None else _rows_2d(targets)
    if y is not None and y.shape[0] != n:
        raise ValueError(f"targets have {y.shape[0]} rows, expected {n}")
    return y


def head_fused_rows(op: int, x, weight, weight_t, targets, target_stats=None, n_rows=None, step=None):
    """``fused_rows`` with the frozen head in front: ``x [1, T, H]`` instead of logits (for callers that reduce the row losses
    themselves; the models take ``head_step_loss`` and ``head_terms_loss``).  Returns ``(row_loss [1, n_rows], argmax_draft,
    argmax_target, lse_target, logits [1, T, Vd])``."""
    n = x.shape[1] if n_rows is None else int(n_rows)
    y = _check_head(x, weight, targets, n)
    t = x.shape[1]
    ks = (None, None) if target_stats is None else (target_stats[0], target_stats[1])
    # (a view, not x[0]: the backward of a select writes the gradient into a zero-filled copy)
    loss, am_d, am_t, lse_t, logits = _HeadFusedLoss.apply(x.reshape(t, x.shape[2]), weight, weight_t, y, op,
                                                           ks[0], ks[1], n, step)
    lead = (1, n)
    return (loss.view(lead), am_d.view(lead), am_t.view(lead), lse_t.view(lead),
            logits.view(1, t, weight.shape[0]))


def fused_rows(op: int, logits, targets, target_stats=None, n_rows=None, step: StepPass | None = None):
    """(row_loss, argmax_draft, argmax_target, lse_target) of one primitive reduction;
    ``n_rows`` restricts ``logits [1, T, V]`` to its first ``n_rows`` rows (``targets`` already
    has that many) without slicing it under autograd; ``step``: see ``StepPass``."""
    if target_stats is None:
        return _FusedLoss.apply(logits, targets, op, None, None, n_rows, step)
    return _FusedLoss.apply(logits, targets, op, target_stats[0], target_stats[1], n_rows, step)


def kl_div_loss(logits, targets):
    return _lib.native().row_loss(OP_KL, logits, targets)


def reverse_kl_div_loss(logits, targets):
    return _lib.native().row_loss(OP_RKL, logits, targets)


def js_div_loss(logits, targets):
    return _lib.native().row_loss(OP_JSD, logits, targets)


def ce_loss(logits, targets):
    return _lib.native().row_loss(OP_CE, logits, targets)


def tv_loss(logits, targets):
    return _lib.native().row_loss(OP_TV, logits, targets)


def neg_log_acceptance_loss(logits, targets):
    """-log(max(1 - tv, 1e-5)) composed on the [B, T] tv rows (losses/fused.py:322-324)."""
    return -torch.log((1.0 - tv_loss(logits, targets)).clamp_min(_NLA_EPS))


def lk_hybrid_loss(logits, targets, eta: float = 3.0):
    """lam*kl + (1-lam)*tv with lam = exp(-eta*stopgrad(1-tv)) (losses/fused.py:327-334)."""
    kl = kl_div_loss(logits, targets)
    tv = tv_loss(logits, targets)
    lam = torch.exp(-eta * (1.0 - tv).detach())
    return lam * kl + (1.0 - lam) * tv


_HIP_LOSS_FN_MAP: dict[str, Callable] = {
    "kl_div": kl_div_loss,
    "rkl": reverse_kl_div_loss,
    "jsd": js_div_loss,
    "ce": ce_loss,
    "tv": tv_loss,
    "nla": neg_log_acceptance_loss,
    "lk_hybrid": lk_hybrid_loss,
}

# which primitive kernel reduction also yields the arg-maxes for a named loss
PRIMITIVE_OP = {"kl_div": OP_KL, "rkl": OP_RKL, "jsd": OP_JSD, "ce": OP_CE, "tv": OP_TV}

_LOSS_FN_MAPS = {"hip": _HIP_LOSS_FN_MAP}


def resolve_loss_config(spec: str, implementation: str = "hip") -> LossConfig:
    """``"kl_div"`` or ``'{"ce": 0.1, "tv": 0.9}'`` -> ``{name: (fn, weight)}`` with the
    error behaviour of losses/utils.py:184-230."""
    try:
        table = _LOSS_FN_MAPS[implementation]
    except KeyError:
        raise ValueError(
            f"Unknown loss implementation '{implementation}'. Choose from: {sorted(_LOSS_FN_MAPS)}"
        ) from None
    if spec in table:
        return {spec: (table[spec], 1.0)}
    try:
        parsed = json.loads(spec)
    except json.JSONDecodeError:
        raise ValueError(
            f"Unknown loss function '{spec}'. Pass a known name ({sorted(table)}) or a JSON dict, "
            'e.g. \'{"ce": 0.1, "tv": 0.9}\'.'
        ) from None
    if not isinstance(parsed, dict) or not parsed:
        raise ValueError(
            "Loss config must be a non-empty JSON dict mapping loss names to weights, "
            f'e.g. \'{{"ce": 0.1, "tv": 0.9}}\'. Got: {spec}'
        )
    out: LossConfig = {}
    for name, weight in parsed.items():
        if name not in table:
            raise ValueError(
                f"Unknown loss function '{name}' in loss config. Choose from: {sorted(table)}"
            )
        if isinstance(weight, bool) or not isinstance(weight, (int, float)):
            raise ValueError(
                f"Loss weight for '{name}' must be a number, got {type(weight).__name__}"
            )
        out[name] = (table[name], float(weight))
    return out


class _LabelCE(torch.autograd.Function):
    """Per-row cross-entropy of ``logits [R, V]`` against integer ``labels [R]`` with an
    ignore index, on the HIP label-CE kernels (one read of the logits in the forward, one
    read + one write in the backward)."""

    @staticmethod
    def forward(ctx, logits2d, labels, ignore_index):
        rows, vocab = logits2d.shape
        dev = logits2d.device
        out = torch.empty(2, rows, device=dev, dtype=torch.float32)
        _lib.call("spx_label_ce_fwd", logits2d, logits2d.stride(0), labels, rows,
                  vocab, _lib.dtype_code(logits2d), int(ignore_index), out[0],
                  out[1], None, _lib.stream_ptr(dev))
        ctx.save_for_backward(logits2d, labels, out[1])
        ctx.ignore_index = int(ignore_index)
        return out[0]

    @staticmethod
    def backward(ctx, grad_rows):
        logits2d, labels, lse = ctx.saved_tensors
        rows, vocab = logits2d.shape
        g = grad_rows.to(torch.float32).contiguous()
        dlogits = torch.empty(rows, vocab, device=logits2d.device, dtype=logits2d.dtype)
        _lib.call("spx_label_ce_bwd", logits2d, logits2d.stride(0), labels,
                  lse, g, rows, vocab, _lib.dtype_code(logits2d),
                  ctx.ignore_index, dlogits, dlogits.stride(0),
                  _lib.stream_ptr(logits2d.device))
        return dlogits, None, None


def label_cross_entropy(logits: torch.Tensor, labels: torch.Tensor, ignore_index: int = -100):
    """``F.cross_entropy(logits.permute(0, 2, 1), labels, ignore_index=..., reduction="none")``
    (models/mtp/core.py:204-216) for ``logits [..., V]`` (bf16 or fp32) and integer ``labels
    [...]``: returns float32 losses of the shape of ``labels``, 0 at ignored positions."""
    if logits.shape[:-1] != labels.shape:
        raise ValueError(f"logits {tuple(logits.shape)} and labels {tuple(labels.shape)} do not match")
    if logits.dtype not in (torch.bfloat16, torch.float32):
        raise _lib.SpxError("label_cross_entropy takes bf16 or fp32 logits")
    x = _rows_2d(logits)
    lab = labels.reshape(-1).to(torch.int64).contiguous()
    return _LabelCE.apply(x, lab, ignore_index).view(labels.shape)


class _HeadLabelCE(torch.autograd.Function):
    """A frozen output head and the label cross-entropy behind it as ONE autograd node:
    ``(x [R, H], weight [V, H], weight_t [H, V], labels [R]) -> (row loss [R] f32, logits [R, V])``.

    What the single node buys is the backward: a position with an ignored label (or a zero
    incoming gradient) has an all-zero logits-gradient row, so the loss backward packs the live
    rows to the front (``spx_label_ce_bwd_packed``) and the input-gradient product runs over
    those rows only (``spx_gemm_bf16_nt_rows``, row count read on the device, no host
    synchronisation); the dead rows of ``dx`` are exact zeros, as they are when the product
    runs over all rows.  The logits come back for the caller's metrics / return value but carry
    no gradient of their own."""

    @staticmethod
    def forward(ctx, x2, weight, weight_t, labels, ignore_index, epilogue_stats=False, room=None):
        from .gemm import gemm_nt_stats, matmul_nt

        ctx.one_pass = False
        one_pass = room is not None and not epilogue_stats  # room: GradientRoom, where the one-read pass takes the rows
        if one_pass:
            logits = matmul_nt(x2, weight)
            packed = room.take(logits)
            if packed is not None:
                ctx.one_pass = True
                rows, vocab = logits.shape
                loss = torch.empty(rows, device=logits.device, dtype=torch.float32)
                lists = torch.empty(2 * rows + 1, device=logits.device, dtype=torch.int32)
                row_map, row_of, count = lists[:rows], lists[rows:2 * rows], lists[2 * rows:]
                _lib.call("spx_label_ce_fwd_grad", logits, logits.stride(0), labels, rows, vocab, int(ignore_index), loss,
                          row_map, count, row_of, packed, vocab, _lib.stream_ptr(logits.device))
                ctx.save_for_backward(packed, row_map, count, weight_t, row_of)
                ctx.mark_non_differentiable(logits)
                ctx.set_materialize_grads(False)
                return loss, logits
        if epilogue_stats:
            # the head product's epilogue leaves every row's log-sum-exp; the loss then reads one
            # element of each row instead of streaming the [rows, V] logits a second time
            logits, lse, _ = gemm_nt_stats(x2, weight, want_argmax=False)
            rows, vocab = logits.shape
            out = torch.empty(2, rows, device=logits.device, dtype=torch.float32)
            out[1] = lse
            _lib.call("spx_label_ce_from_lse", logits, logits.stride(0), labels, rows,
                      vocab, _lib.dtype_code(logits), int(ignore_index), out[1], out[0],
                      _lib.stream_ptr(logits.device))
        else:
            if not one_pass:
                logits = matmul_nt(x2, weight)
            rows, vocab = logits.shape
            out = torch.empty(2, rows, device=logits.device, dtype=torch.float32)
            _lib.call("spx_label_ce_fwd", logits, logits.stride(0), labels, rows,
                      vocab, _lib.dtype_code(logits), int(ignore_index), out[0],
                      out[1], None, _lib.stream_ptr(logits.device))
        ctx.save_for_backward(logits, labels, out[1], weight_t)
        ctx.ignore_index = int(ignore_index)
        ctx.mark_non_differentiable(logits)
        ctx.set_materialize_grads(False)  # no [rows, V] zeros for the logits, which carry no gradient
        return out[0], logits

    @staticmethod
    def backward(ctx, grad_rows, _grad_logits):
        from .gemm import matmul_nt, rows_graded

        if grad_rows is None:
            return (None,) * 7
        if ctx.one_pass:
            packed, row_map, count, weight_t, row_of = ctx.saved_tensors
            g = grad_rows.to(torch.float32).contiguous()
            one = torch.ones((), device=g.device, dtype=torch.float32)
            dx = rows_graded(packed, weight_t, count, row_of, g, one, 1.0)
            # (a row whose incoming gradient is zero has a gradient of zero, whatever its logits are)
            dx = _unpack_rows(dx, torch.where(g == 0, -1, row_map), row_map.numel())
            return (dx,) + (None,) * 6

        logits, labels, lse, weight_t = ctx.saved_tensors
        rows, vocab = logits.shape
        g = grad_rows.to(torch.float32).contiguous()
        row_map, count = _packed_row_map(g, labels, ctx.ignore_index)
        packed = torch.empty(rows, vocab, device=logits.device, dtype=logits.dtype)
        _lib.call("spx_label_ce_bwd_packed", logits, logits.stride(0), labels,
                  lse, g, rows, vocab, _lib.dtype_code(logits), ctx.ignore_index,
                  row_map, packed, packed.stride(0),
                  _lib.stream_ptr(logits.device))
        dx_packed = matmul_nt(packed, weight_t, m_live=count)
        return (_unpack_rows(dx_packed, row_map, rows),) + (None,) * 6


def _label_one_pass(x2, weight) -> bool:
    """Whether the row pass of the frozen-head cross-entropy leaves the logits gradient behind
    (``spx_label_ce_fwd_grad``): rows that fit a workgroup's registers and give every thread eight chunks at least."""
    vocab = weight.shape[0]
    return (HEAD_LOSS_ONE_PASS and torch.is_grad_enabled() and x2.requires_grad and vocab % 8 == 0 and 65536 <= vocab <= 155648
            and 0 < x2.shape[0] < 1 << 31)


# of the memory that is available at a call, what the logits gradients of this call and of those still to come in the same
# forward may take from their forward to their backward.  The logits of the calls to come take as much again, and half is
# left for what the two-pass form needs as well: the activations of the layers in between (of a row, 60 KB beside 300 KB of
# logits at 2048 -> 151936 and 250 KB beside 130 KB at 5120 -> 65536, the widest for its logits), and the backward
LABEL_GRADIENT_SHARE = 1 / 4


def _available_memory(device) -> int:
    """Bytes that this process can still allocate: free on the card or held by the allocator, within the process's share.
    (10 us, 90 behind a full queue; no synchronisation, and no launch that a capture would refuse.)"""
    free, total = torch.cuda.mem_get_info(device)
    try:
        stats = torch.cuda.memory_stats_as_nested_dict(device)
        held, used = (stats[f"{kind}_bytes"]["all"]["current"] for kind in ("reserved", "allocated"))
    except (KeyError, RuntimeError):  # an allocator without statistics
        return free
    return min(free + held - used, int(total * torch.cuda.get_per_process_memory_fraction(device)) - used)


class GradientRoom:
    """Where the logits gradients of the head cross-entropies of one forward, ``calls`` of them, wait for its backward."""

    def __init__(self, calls: int = 1):
        self.calls = calls

    def take(self, logits):
        """The place for one, or None: it is made in the backward then, from the logits."""
        left, self.calls = max(self.calls, 1), self.calls - 1
        if left * logits.numel() * 2 > LABEL_GRADIENT_SHARE * _available_memory(logits.device):
            return None
        try:
            return torch.empty_like(logits)
        except torch.OutOfMemoryError:
            return None


# Whether the frozen-head cross-entropy takes its row statistics from the head product's epilogue
# (spx_gemm_bf16_nt_stats, log-sum-exp only) instead of a streaming pass over the logits
# (spx_label_ce_fwd).  The epilogue's exponentials hold the matrix pipe up for as long as the streaming pass takes
# where live rows are 70 %: one iteration of the MTP head (three steps, 32760 rows x 2048 -> 151936) 186.3 ms with
# the epilogue, 185.6 streaming; 2 x 4096 rows 38.6 and 38.2; 2000 rows, two steps 7.64 and 7.45; 600 rows 5.38 and 5.29.
HEAD_CE_EPILOGUE_STATS = False


def head_label_cross_entropy(x: torch.Tensor, weight: torch.Tensor, weight_t: torch.Tensor,
                             labels: torch.Tensor, ignore_index: int = -100,
                             epilogue_stats: bool | None = None, room: GradientRoom | None = None):
    """``logits = x @ weight.T`` and ``F.cross_entropy(logits, labels, ignore_index=...,
    reduction="none")`` (models/mtp/core.py:190-216) for a FROZEN ``weight [V, H]`` whose
    transpose ``weight_t [H, V]`` the caller keeps: returns ``(loss [...] f32, logits [..., V])``.
    Gradient flows to ``x`` through the loss only; the returned logits are detached.  ``room``: one for all calls of a forward
    (None: this is the only one)."""
    if x.dtype != torch.bfloat16 or weight.dtype != torch.bfloat16 or weight_t.dtype != torch.bfloat16:
        raise _lib.SpxError("head_label_cross_entropy takes bf16 operands")
    if weight.requires_grad:
        raise ValueError("head_label_cross_entropy is for a frozen head (no weight gradient is produced)")
    if x.shape[:-1] != labels.shape:
        raise ValueError(f"x {tuple(x.shape)} and labels {tuple(labels.shape)} do not match")
    if weight_t.shape != (weight.shape[1], weight.shape[0]) or not weight_t.is_contiguous():
        raise ValueError("weight_t must be the contiguous transpose of weight")
    x2 = x.reshape(-1, x.shape[-1])
    lab = labels.reshape(-1).to(torch.int64).contiguous()
    if epilogue_stats is None:
        epilogue_stats = HEAD_CE_EPILOGUE_STATS
    room = (room or GradientRoom()) if _label_one_pass(x2, weight) else None
    loss, logits = _HeadLabelCE.apply(x2, weight, weight_t, lab, ignore_index, bool(epilogue_stats), room)
    return loss.view(labels.shape), logits.view(*labels.shape, weight.shape[0])


def vocab_gather(full_logits: torch.Tensor, d2t: torch.Tensor) -> torch.Tensor:
    """``full_logits[..., i + d2t[i]]`` on the device: verifier logits over the target
    vocabulary restricted to the draft vocabulary (the gather form of the t2d row-slice,
    model.py:161-169, with the offset table of train/vocab_mapping.py:86-96)."""
    x = _rows_2d(full_logits)
    rows, vt = x.shape
    vd = d2t.numel()
    d2t = d2t.to(device=x.device, dtype=torch.int64).contiguous()
    out = torch.empty(rows, vd, device=x.device, dtype=x.dtype)
    done = 0
    while done < rows:  # the gather grid carries rows in its y dimension
        n = min(rows - done, 65535)
        xs, os_ = x[done:done + n], out[done:done + n]
        _lib.call("spx_vocab_gather", xs, x.stride(0), d2t, os_,
                  out.stride(0), n, vd, vt, _lib.dtype_code(x), _lib.stream_ptr(x.device))
        done += n
    return out.view(*full_logits.shape[:-1], vd)
