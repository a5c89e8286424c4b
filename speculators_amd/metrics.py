"""Per-step loss and acceptance metrics on the device.

Drop-in replacements, with identical metric keys and the identical in-place
mutation of ``prev_correct``, for
  * ``compute_metrics`` of EAGLE3 (models/eagle3/metrics.py:51-119) and
  * ``compute_metrics`` of DFlash (models/dflash/metrics.py:20-108).
The row losses and both arg-maxes come out of one pass of the fused loss
kernel; the masked mean, the acceptance chain and the counts are one more
single-workgroup kernel.  Nothing of size ``[T, V]`` is ever created here.
"""

from __future__ import annotations

import numpy as np
import torch

from . import _lib
from . import losses as L


def _as_mask(t: torch.Tensor) -> torch.Tensor:
    """1-D unit-stride view of a ``[1, n]`` mask (its dtype is kept)."""
    t = t.reshape(-1)
    return t if t.stride(0) == 1 else t.contiguous()


class _StepReduce(torch.autograd.Function):
    """(row_loss [n] f32, total_in) -> total_in + factor * weighted masked mean (0-d); also fills the mean's
    ``out`` and, where the loss pass has not done the acceptance chain (no ``counts``), leaves it out:
    d/d row_loss = factor * row_weight."""

    @staticmethod
    def forward(ctx, row_loss, total_in, am_d, am_t, mean, counts):
        shape = row_loss.shape
        total, row_weight = mean.reduce(row_loss.reshape(-1).contiguous(), am_d, am_t, counts, total_in)
        ctx.save_for_backward(row_weight)
        ctx.shape, ctx.factor = shape, mean.factor
        return total

    @staticmethod
    def backward(ctx, g):
        (row_weight,) = ctx.saved_tensors
        scaled = g if ctx.factor == 1.0 else g * ctx.factor
        return (row_weight * scaled).view(ctx.shape), g if ctx.needs_input_grad[1] else None, None, None, None, None


class TargetGather:
    """Full-vocabulary verifier logits (``[1, T, Vt]``) with the ``d2t`` offset table, standing
    where ``compute_metrics`` takes the targets.  The first TTT step reads its target rows
    THROUGH the table inside the loss pass (no gather kernel, no ``[T, Vd]`` copy made first) and
    leaves the draft-vocabulary rows in ``compact`` (``[1, T, Vd]``), which the later steps and the
    backward stream."""

    def __init__(self, full_logits: torch.Tensor, d2t: torch.Tensor):
        if full_logits.dim() != 3 or full_logits.shape[0] != 1:
            raise ValueError("verifier logits must be [1, T, Vt] (the packed batch layout)")
        self.full = full_logits
        self.d2t = d2t.to(torch.int64).contiguous()
        self.compact = None

    def materialize(self) -> torch.Tensor:
        if self.compact is None:
            self.compact = L.vocab_gather(self.full, self.d2t)
        return self.compact


class VerifierHead:
    """The frozen verifier head (``verifier_lm_head(verifier_norm(h))``, models/eagle3/core.py:250-253)
    applied lazily, standing where ``compute_metrics`` takes the targets.  A cross-entropy loss needs
    nothing of the target logits but their row arg-max (losses/eager.py ``ce_loss``), and the acceptance
    metrics need the same: with that loss alone the head product is reduced to per-row statistics in its
    own epilogue (``gemm.gemm_nt_stats(store=False)``) and the ``[T, Vd]`` target logits are never
    written or read.  Any other loss gets them the ordinary way (``materialize``)."""

    def __init__(self, x: torch.Tensor, weight: torch.Tensor):
        if x.dim() != 3 or x.shape[0] != 1:
            raise ValueError("verifier hidden states must be [1, T, H] (the packed batch layout)")
        self.x, self.weight = x, weight
        self.logits = None

    def materialize(self) -> torch.Tensor:
        from . import gemm

        if self.logits is None:
            self.logits = gemm.matmul_nt(self.x[0], self.weight).view(1, self.x.shape[1], self.weight.shape[0])
        return self.logits

    def stats(self):
        """(lse [T] f32, argmax [T] i32) of the target rows; the rows themselves are not stored.  The
        cross-entropy reads the arg-max only: the log-sum-exp is not computed (zeros stand in)."""
        from . import gemm

        _, _, am = gemm.gemm_nt_stats(self.x[0], self.weight, store=False, want_lse=False)
        return torch.zeros(am.shape, device=am.device, dtype=torch.float32), am


def _step_views(logits, targets, loss_mask, prev_correct, ttt_step):
    """align_for_step (models/eagle3/metrics.py:16-48): views only."""
    n = logits.shape[1] - ttt_step
    return (
        logits[:, :n],
        None if targets is None else targets[:, ttt_step:],
        None if loss_mask is None else loss_mask[:, ttt_step:],
        None if prev_correct is None else prev_correct[:, :n],
    )


class Head:
    """The frozen ``lm_head`` applied lazily: ``compute_metrics`` takes this in place of the logits
    and, when the loss is of fused HIP reductions, runs head and loss as ONE autograd node (the
    backward then skips the rows the loss mask removes in the head's input-gradient product,
    ``losses.head_step_loss``, ``losses.head_terms_loss``); otherwise the logits are made the ordinary way.  Either way
    ``.logits`` holds them afterwards (``[1, T, Vd]``)."""

    def __init__(self, x, weight, weight_t):
        self.x, self.weight, self.weight_t = x, weight, weight_t
        self.logits = None

    def materialize(self):
        from . import gemm

        if self.logits is None:
            self.logits = gemm.linear(self.x, self.weight, self.weight_t)
        return self.logits


def _flat_prev(s_prev):
    if s_prev is None:
        return None
    prev1 = s_prev.reshape(-1)
    if prev1.stride(0) != 1:
        raise ValueError("prev_correct must be contiguous (it is updated in place)")
    return prev1


def _terms_step(head, targets, loss_mask, prev_correct, ttt_step, decay, loss_config, cache, return_pred, total_in,
                return_tokens):
    """``compute_metrics`` with the whole loss in one row pass behind the head (``losses.head_terms_loss``), or None where
    that does not take it."""
    n = head.x.shape[1] - ttt_step
    gather = targets if isinstance(targets, TargetGather) and targets.compact is None and ttt_step == 0 else None
    if isinstance(targets, TargetGather):
        rows = targets.full if gather is not None else targets.compact
    elif isinstance(targets, VerifierHead):
        rows = targets.weight if targets.logits is None else targets.logits  # (its logits are bf16 rows of that width)
        rows = rows if targets.logits is not None else rows.new_empty(0, rows.shape[0])
    else:
        rows = targets
    if (head.x.shape[0] != 1 or rows is None or head.x.dtype != torch.bfloat16
            or not L.terms_fit(loss_config, head.weight, rows, None if gather is None else gather.d2t,
                               None if loss_mask is None else loss_mask[:, ttt_step:], n)):
        return None
    if gather is None and not isinstance(targets, torch.Tensor):
        rows = targets.materialize()
    _, s_targets, s_mask, s_prev = _step_views(head.x, rows, loss_mask, prev_correct, ttt_step)
    out = torch.empty(18, device=head.x.device, dtype=torch.float32)
    known = None
    if cache is not None and cache.get("kl") is not None and gather is None:
        known = (cache["kl"][0][ttt_step:], cache["kl"][1][ttt_step:])
    step = L.StepPass(mask=_as_mask(s_mask), prev=_flat_prev(s_prev))
    total, am_d, am_t, lse_t, head.logits = L.head_terms_loss(
        loss_config, head.x, head.weight, head.weight_t, s_targets, None if gather is None else gather.d2t, known, n, step,
        float(np.float32(decay) ** np.float32(ttt_step)), out, total_in)
    if gather is not None:
        gather.compact = step.gathered.view(1, n, step.gathered.shape[-1])
    if cache is not None and known is None and ttt_step == 0:
        cache["kl"] = (lse_t, am_t)
    m = {f"loss_{ttt_step}_sum": out[6], f"loss_{ttt_step}_total": out[7]}
    if len(loss_config) > 1:
        for name in loss_config:
            op = L.PRIMITIVE_OP[name]
            m[f"{name}_loss_{ttt_step}_sum"] = out[8 + op]
            m[f"{name}_loss_{ttt_step}_total"] = out[13 + op]
    m[f"full_acc_{ttt_step}_sum"] = out[1]
    m[f"full_acc_{ttt_step}_total"] = out[2]
    m[f"cond_acc_{ttt_step}_sum"] = out[3]
    m[f"cond_acc_{ttt_step}_total"] = out[4]
    if return_tokens:
        return total, m, row_tokens(am_d, head.logits.detach()[0, n:])
    return (total, m, am_d) if return_pred else (total, m)


class TTTSteps:
    """``compute_metrics`` of all steps of a TTT loop at once, where one node takes them (``losses.head_steps_loss``):
    terms of kl, ce and tv over bf16 rows, with a loss mask.  ``add`` a step's head input, ``finish`` behind the last."""

    def __init__(self, config, steps, targets, loss_mask, prev_correct, decay):
        self.config, self.steps, self.targets = config, steps, targets
        self.mask, self.prev = loss_mask, prev_correct
        self.weights = [float(np.float32(decay) ** np.float32(k)) for k in range(steps)]
        ops = {L.PRIMITIVE_OP[name]: float(w) for name, (_, w) in config.items()}
        self.op = next(iter(ops))
        self.factor = ops[self.op]
        # one kl or ce has a form of its own
        self.terms = None if len(ops) == 1 and self.op != L.OP_TV else tuple(ops.get(op) for op in range(5))
        self.xs = []

    @staticmethod
    def take(x, weight, targets, loss_mask, prev_correct, steps, decay, loss_config):
        """The steps behind ``x`` (the first one's head input), or None where ``compute_metrics`` has to take them."""
        if loss_config is None:
            loss_config = {"kl_div": (L.kl_div_loss, 1.0)}
        if (compute_metrics is not _own_compute_metrics or loss_mask is None or not loss_config
                or not L.steps_fit(loss_config, steps, x, weight, loss_mask)):
            return None
        shape, vocab = tuple(x.shape[:-1]), weight.shape[0]
        if tuple(loss_mask.shape) != shape or tuple(prev_correct.shape) != shape:
            return None
        if isinstance(targets, VerifierHead):  # (its rows are bf16, contiguous, of its weight's width)
            fits = targets.x.shape[1] == shape[1] and targets.weight.shape[0] == vocab and targets.weight.dtype == torch.bfloat16
        elif isinstance(targets, TargetGather):
            fits = (targets.full.shape[:2] == shape and targets.full.dtype == torch.bfloat16 and targets.d2t.numel() == vocab
                    and targets.compact is None)
        else:
            fits = targets.dim() == 3 and targets.shape[0] == 1 and L.steps_rows_fit(targets[0], shape[1], vocab)
        return TTTSteps(loss_config, steps, targets, _as_mask(loss_mask), _flat_prev(prev_correct), decay) if fits else None

    def add(self, x):
        self.xs.append(x)

    def finish(self, weight, weight_t, logits=None):
        """``(loss, metrics, draft tokens of every step [1, T])``; ``logits``: a list that receives every step's."""
        rows = argmax = None
        targets = self.targets
        if isinstance(targets, VerifierHead) and self.terms is None and self.op == L.OP_CE and targets.logits is None:
            argmax = targets.stats()[1]  # no target row exists
        else:
            rows = (targets if isinstance(targets, torch.Tensor) else targets.materialize())[0]
        kept = None if logits is None else []
        # (the pass that gathers a first step's rows for several terms knows their statistics: masked rows are not formed)
        run = L.HeadSteps(self.op, self.weights, self.factor if self.terms is None else 1.0, self.mask, self.prev, rows, argmax, kept,
                          self.terms, not (self.terms and isinstance(targets, TargetGather)))
        loss = L.head_steps_loss(run, weight, weight_t, self.xs)
        if logits is not None:
            logits += [x.view(1, *x.shape) for x in kept]
        m = {}
        for k in range(self.steps):
            out = run.scalars[k]
            m[f"loss_{k}_sum"], m[f"loss_{k}_total"] = out[6], out[7]
            if len(self.config) > 1:
                for name in self.config:
                    op = L.PRIMITIVE_OP[name]
                    m[f"{name}_loss_{k}_sum"], m[f"{name}_loss_{k}_total"] = out[8 + op], out[13 + op]
            m[f"full_acc_{k}_sum"], m[f"full_acc_{k}_total"] = out[1], out[2]
            m[f"cond_acc_{k}_sum"], m[f"cond_acc_{k}_total"] = out[3], out[4]
        return loss, m, list(run.tokens.split(1))


def compute_metrics(logits, targets, loss_mask, prev_correct, ttt_step: int,
                    ttt_step_loss_decay: float, loss_config: L.LossConfig | None = None,
                    target_stats_cache: dict | None = None, return_pred: bool = False,
                    total_in: torch.Tensor | None = None, return_tokens: bool = False):
    """EAGLE3 per-step loss + metrics; same contract as models/eagle3/metrics.py:51-119.

    ``prev_correct`` (any mask dtype) is updated in place.  Returns
    ``(loss 0-d, metrics dict of 0-d tensors)``.

    Optional extras beyond the reference contract: ``target_stats_cache`` (a dict the
    caller keeps across the TTT steps of ONE forward) lets steps >= 1 reuse the verifier
    rows' log-sum-exp / arg-max computed at step 0 (``targets`` is the same tensor at every
    step, only shifted); ``return_pred=True`` also returns the draft arg-max of the aligned
    rows (int32 ``[T - ttt_step]``), ``return_tokens=True`` that of all rows (int64 ``[1, T]``: the last ``ttt_step``
    rows have no target); ``total_in`` (0-d) is added to the returned loss, not to its metric.
    """
    if loss_config is None:
        loss_config = {"kl_div": (L.kl_div_loss, 1.0)}
    head = None
    if isinstance(logits, Head):
        # one node for head + loss: a loss of one streaming reduction in its own form, the others as weighted terms
        (name0, (fn0, _w0)), = list(loss_config.items())[:1]
        frozen = logits.x.requires_grad and not logits.weight.requires_grad and logits.weight_t is not None
        if frozen and (len(loss_config) > 1 or name0 not in ("kl_div", "ce")):
            done = _terms_step(logits, targets, loss_mask, prev_correct, ttt_step, ttt_step_loss_decay, loss_config,
                               target_stats_cache, return_pred, total_in, return_tokens)
            if done is not None:
                return done
        single = (frozen and len(loss_config) == 1 and name0 in L.PRIMITIVE_OP
                  and fn0 is L._HIP_LOSS_FN_MAP.get(name0))
        if single:
            head = logits
            logits = head.x[:, :, :0].detach()  # shape carrier only
        else:
            logits = logits.materialize()
    if logits.shape[0] != 1:
        raise ValueError("the packed batch layout has batch size 1 (train/data.py:306-393)")
    gather = None
    if isinstance(targets, TargetGather):
        name0, (fn0, _) = next(iter(loss_config.items()))
        if (targets.compact is None and ttt_step == 0 and name0 in L.PRIMITIVE_OP
                and fn0 is L._HIP_LOSS_FN_MAP.get(name0)):
            gather, targets = targets, targets.full  # read through d2t inside the first loss pass
        else:
            targets = targets.materialize()
    if isinstance(targets, VerifierHead):
        (name0, (fn0, _w0)), = list(loss_config.items())[:1]
        ce_only = (len(loss_config) == 1 and name0 == "ce" and fn0 is L._HIP_LOSS_FN_MAP.get("ce")
                   and target_stats_cache is not None and targets.logits is None)
        if ce_only:
            if "ce" not in target_stats_cache:
                target_stats_cache["ce"] = targets.stats()
            targets = None  # every step reads the statistics; no target row exists
        else:
            targets = targets.materialize()
    s_logits, s_targets, s_mask, s_prev = _step_views(
        logits, targets, loss_mask, prev_correct, ttt_step)
    dev = logits.device
    # gamma ** step evaluated in fp32 like exp_loss_decay on a float tensor
    # (losses/utils.py:51-61)
    weight = float(np.float32(ttt_step_loss_decay) ** np.float32(ttt_step))

    mask1 = None if s_mask is None else _as_mask(s_mask)
    prev1 = _flat_prev(s_prev)

    multi = len(loss_config) > 1
    # (one term: its mean goes straight onto the loss so far; several: onto each other first)
    total = None if multi else total_in
    terms = {}
    first_out = None
    counts = None
    for ti, (name, (fn, w)) in enumerate(loss_config.items()):
        out = torch.empty(8, device=dev, dtype=torch.float32)
        mean = L.MeanTerm(mask1, weight, float(w), out)
        op = L.PRIMITIVE_OP.get(name)
        step = None
        if ti == 0:
            # the first term's row pass also gathers the targets (first step of a TargetGather)
            # and advances the acceptance chain
            if head is None:
                counts = torch.zeros(3, device=dev, dtype=torch.int32)
            # (a row the mask removes has weight zero in the masked mean below: the head + loss node may
            # write the logits gradient of the other rows in the same pass)
            step = L.StepPass(d2t=gather.d2t if gather is not None else None, mask=mask1, prev=prev1,
                              counts=counts, grad_in_pass=head is not None and mask1 is not None)
        elif gather is not None:
            s_targets = gather.compact
        if fn is L._HIP_LOSS_FN_MAP.get(name) and op is not None:
            known = None
            if target_stats_cache is not None and op in (L.OP_KL, L.OP_CE) and gather is None:
                full = target_stats_cache.get("kl" if op == L.OP_KL else "ce")
                if full is None and op == L.OP_CE:
                    full = target_stats_cache.get("kl")  # the arg-max is all ce needs
                if full is not None:
                    known = (full[0][ttt_step:], full[1][ttt_step:])
            # the full logits go in with a row count: see _FusedLoss.forward
            if head is not None:
                total, am_d, am_t, lse_t, head.logits = L.head_step_loss(
                    op, head.x, head.weight, head.weight_t, s_targets, known, s_logits.shape[1], step, mean, total)
            else:
                rows, am_d, am_t, lse_t = L.fused_rows(op, logits, s_targets, known,
                                                       n_rows=s_logits.shape[1], step=step)
            if step is not None and step.gathered is not None:
                gather.compact = step.gathered.view(1, -1, step.gathered.shape[-1])
            if (target_stats_cache is not None and known is None and ttt_step == 0
                    and op in (L.OP_KL, L.OP_CE)):
                target_stats_cache["kl" if op == L.OP_KL else "ce"] = (
                    lse_t.reshape(-1), am_t.reshape(-1))
        else:
            rows = fn(s_logits, s_targets)
            _, am_d, am_t, _ = L.fused_rows(L.OP_CE, s_logits.detach(), s_targets, step=step)
        if ti == 0:
            pred = am_d.reshape(-1)
        # only the first term advances the acceptance chain (inside its row pass)
        if head is None:
            total = _StepReduce.apply(rows.reshape(-1), total, am_d.reshape(-1), am_t.reshape(-1), mean,
                                      counts if ti == 0 else None)
        if ti == 0:
            first_out = out
        if multi:
            terms[f"{name}_loss"] = out[0]

    one = first_out[7]
    if multi:
        m = {f"loss_{ttt_step}_sum": total.detach().clone(), f"loss_{ttt_step}_total": one}
        if total_in is not None:
            total = total_in + total
    else:
        m = {f"loss_{ttt_step}_sum": first_out[6], f"loss_{ttt_step}_total": one}
    for tname, tval in terms.items():
        m[f"{tname}_{ttt_step}_sum"] = tval
        m[f"{tname}_{ttt_step}_total"] = one.clone()
    m[f"full_acc_{ttt_step}_sum"] = first_out[1]
    m[f"full_acc_{ttt_step}_total"] = first_out[2]
    m[f"cond_acc_{ttt_step}_sum"] = first_out[3]
    m[f"cond_acc_{ttt_step}_total"] = first_out[4]
    if return_tokens:
        return total, m, row_tokens(pred, (logits if head is None else head.logits).detach()[0, s_logits.shape[1]:])
    if return_pred:
        return total, m, pred
    return total, m


_own_compute_metrics = compute_metrics  # (a replaced one is called, step by step)


def row_tokens(known, rows: torch.Tensor) -> torch.Tensor:
    """int64 ``[1, n + tail]``: the arg-maxes ``known`` (int32 ``[n]`` or None) and those of ``rows [tail, V]``."""
    n = 0 if known is None else known.numel()
    rows = L._rows_2d(rows)
    tail, vocab = rows.shape
    out = torch.empty(1, n + tail, device=rows.device, dtype=torch.int64)
    _lib.call("spx_row_tokens", known, n, rows if tail else None, rows.stride(0), tail, vocab, _lib.dtype_code(rows),
              out, _lib.stream_ptr(rows.device))
    return out


def argmax_rows(logits: torch.Tensor) -> torch.Tensor:
    """First-index arg-max over the last axis as int64."""
    return row_tokens(None, L._rows_2d(logits)).view(logits.shape[:-1])


class _BlockReduce(torch.autograd.Function):
    """(row_loss [n] f32, total_in) -> total_in + the term (``losses.BlockTerm``); d / d row_loss = factor * row_weight."""

    @staticmethod
    def forward(ctx, row_loss, total_in, am_d, am_t, term):
        total, row_weight = term.reduce(row_loss.reshape(-1).contiguous(), am_d, am_t, None, total_in)
        ctx.save_for_backward(row_weight)
        ctx.shape, ctx.factor = row_loss.shape, term.factor
        return total

    @staticmethod
    def backward(ctx, g):
        (row_weight,) = ctx.saved_tensors
        scaled = g if ctx.factor == 1.0 else g * ctx.factor
        return (row_weight * scaled).view(ctx.shape), g if ctx.needs_input_grad[1] else None, None, None, None


def dflash_loss_decay(pos_idx: torch.Tensor, gamma: float, sample_from_anchor: bool = False):
    """Per-slot weight of losses/utils.py:17-48 (a [block_size]-periodic vector)."""
    pos = pos_idx.to(torch.float32)
    if sample_from_anchor:
        return torch.exp(-pos / gamma)
    w = torch.exp(-(pos - 1.0).clamp_min(0.0) / gamma)
    return torch.where(pos == 0, torch.zeros_like(w), w)


def dpace_loss_decay(row_ce: torch.Tensor, loss_mask: torch.Tensor, block_size: int,
                     dpace_alpha: float) -> torch.Tensor:
    """D-PACE weight from masked CE row losses (losses/utils.py:64-112); no gradient."""
    with torch.no_grad():
        n = row_ce.numel()
        if n % block_size != 0:
            raise ValueError(f"q.shape[1] ({n}) must be divisible by block_size ({block_size})")
        conf = torch.exp(-row_ce.float()).reshape(n // block_size, block_size)
        m = loss_mask.reshape(n // block_size, block_size).to(conf.dtype)
        s = torch.where(m > 0, (1.0 - dpace_alpha) * conf + dpace_alpha, torch.ones_like(conf))
        prefix = torch.cumprod(s, dim=-1) * m
        suffix = torch.flip(torch.cumsum(torch.flip(prefix, dims=[-1]), dim=-1), dims=[-1])
        return (suffix * m).reshape(-1)


def dflash_compute_metrics(logits, targets, loss_mask, block_size: int = 1, gamma: float = 4.0,
                           loss_config: L.LossConfig | None = None,
                           per_position_loss_weight: str = "fixed-exp-decay",
                           dpace_alpha: float = 0.5, sample_from_anchor: bool = False):
    """DFlash loss + per-slot accuracy + EAL; contract of models/dflash/metrics.py:20-108.
    ``logits`` may be a ``Head`` (see ``compute_metrics``)."""
    if loss_config is None:
        loss_config = {"kl_div": (L.kl_div_loss, 1.0)}
    head = None
    if isinstance(logits, Head):
        (name0, (fn0, _w0)), = list(loss_config.items())[:1]
        if (len(loss_config) == 1 and name0 in L.PRIMITIVE_OP and fn0 is L._HIP_LOSS_FN_MAP.get(name0)
                and logits.x.requires_grad and not logits.weight.requires_grad
                and logits.weight_t is not None):
            head = logits
            logits = torch.empty(1, head.x.shape[1], 0, device=head.x.device)  # shape carrier only
        else:
            logits = logits.materialize()
    dev = logits.device
    mask1 = _as_mask(loss_mask)
    total = first = None
    terms = {}
    for ti, (name, (fn, w)) in enumerate(loss_config.items()):
        op = L.PRIMITIVE_OP.get(name)
        out = torch.empty(9 + 2 * block_size, device=dev, dtype=torch.float32)
        dpace = (lambda rows: dpace_loss_decay(rows, mask1, block_size, dpace_alpha)
                 ) if per_position_loss_weight == "dpace" else None
        term = L.BlockTerm(mask1, block_size, gamma, sample_from_anchor, float(w), out, dpace)
        if head is not None:
            total, _, _, _, head.logits = L.head_step_loss(
                op, head.x, head.weight, head.weight_t, targets, None, head.x.shape[1],
                L.StepPass(mask=mask1, grad_in_pass=True), term, total)
        else:
            if fn is L._HIP_LOSS_FN_MAP.get(name) and op is not None:
                rows, am_d, am_t, _ = L.fused_rows(op, logits, targets)
            else:
                rows = fn(logits, targets)
                _, am_d, am_t, _ = L.fused_rows(L.OP_CE, logits.detach(), targets)
            total = _BlockReduce.apply(rows.reshape(-1), total, am_d.reshape(-1), am_t.reshape(-1), term)
        if ti == 0:
            first = out
        if len(loss_config) > 1:
            terms[f"{name}_loss"] = out[0], out[6]

    one = first[7]
    m = {"loss_sum": out[2], "loss_total": one}
    for tname, (tval, tone) in terms.items():
        m[f"{tname}_sum"] = tval
        m[f"{tname}_total"] = tone
    m["full_acc_sum"] = first[3]
    m["full_acc_total"] = first[4]
    m["eal_sum"] = first[5]
    m["eal_total"] = first[8]
    for s in range(0 if sample_from_anchor else 1, block_size):
        m[f"position_{s}_acc_sum"] = first[9 + s]
        m[f"position_{s}_acc_total"] = first[9 + block_size + s]
    return total, m
