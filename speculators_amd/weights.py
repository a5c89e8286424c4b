"""Compute copies of the parameters for one forward / backward.

The kernels compute in bf16.  The parameters may be bf16 (the whole model cast, the regime of
the reference's integration tests, tests/integration/conftest.py:130,165) or fp32 master weights
under ``torch.autocast(dtype=torch.bfloat16)`` (the regime of the reference's trainer,
train/trainer.py:459-465, train/config/schema.py:221-226).  Either way every weight the forward
touches is *staged* once per forward:

  * trainable weights go through one autograd node (``_Stage``) that casts to bf16 and, for
    projections that share their input (q/k/v, gate/up), concatenates them row-wise so they run as
    one product.  The weight gradient comes back through that node, so ``torch.autograd.grad``,
    tensor hooks and post-accumulate-grad hooks see it like any other gradient, and it is cast to
    the parameter's dtype there (fp32 for master weights);
  * a weight that is applied several times in one forward (once per TTT step) does not hand
    autograd one weight-sized gradient per use, and its gradient is not summed over the uses in
    memory either: the inputs ``X_j`` of its uses lie one after the other in ONE buffer
    (``Staged.x_slot``: the kernel that produces an input writes it there) and so do the output
    gradients ``dY_j`` of the backward, so that the weight gradient of all uses is ONE product
    ``[dY_0; dY_1; ...]^T [X_0; X_1; ...]`` with the contraction running over ``uses * T`` rows
    (``spx_gemm_bf16_tn_f32``): the sum over the uses happens in the MFMA accumulators, in fp32,
    and the gradient is written once.  That product runs in the staging node's backward, which
    autograd calls after every use has run its own.  The node has a second, fp32 output of the
    weight's shape that occupies no memory (``Staged.token``, one element expanded); the
    products take it as their differentiable input, and the first one to run its backward
    returns an equally empty marker for it so that the node is reached.  A use whose input
    is not in the buffer (nobody asked for the slot, or it was full) is added by a product of
    its own (accumulating in fp32).  The weights of a layer are staged by one node
    (``WeightStager.get_all``), so that their products are one launch.  The nodes hold what the uses
    left behind (``_Uses``) and not the ``Staged``, whose token leads back to the node: a cycle
    that Python's collector does not see through where a node has several tokens;
  * frozen weights (``lm_head``, ``verifier_lm_head``, ``embed_tokens``) are
    cast (and transposed where the backward needs it) once and kept until the parameter changes:
    the key is ``(data_ptr, _version, dtype)``; ``WeightStager.invalidate()`` drops every kept
    copy, and the models call it from ``train()`` / ``eval()`` and ``load_state_dict`` so that a
    write through ``param.data`` (which does not bump ``_version``) is picked up at those points.
    Frozen norm gains are cast by every forward: a cast of a few KB is no reason to miss such a write.
"""

from __future__ import annotations

import torch

from . import _lib


def _autocast_bf16(device_type: str = "cuda") -> bool:
    return torch.is_autocast_enabled(device_type) and torch.get_autocast_dtype(device_type) == torch.bfloat16


def compute_input(x: torch.Tensor) -> torch.Tensor:
    """An activation input in the compute dtype: bf16 as is; fp32 cast to bf16 under bf16 autocast
    (what the first ``nn.Linear`` of the reference does to it there); anything else is refused."""
    if x.dtype == torch.bfloat16:
        return x
    if x.dtype == torch.float32 and _autocast_bf16(x.device.type):
        return x.to(torch.bfloat16)
    raise RuntimeError(
        "the HIP draft path computes in bf16: cast the model and its inputs to bfloat16, or keep "
        "fp32 master weights and run the forward under torch.autocast(dtype=torch.bfloat16)")


def _check_param_dtype(p: torch.Tensor):
    if p.dtype == torch.bfloat16:
        return
    if p.dtype == torch.float32 and _autocast_bf16(p.device.type):
        return
    raise RuntimeError(
        "the HIP draft path computes in bf16: cast the model to bfloat16, or keep fp32 master "
        "weights and run the forward under torch.autocast(dtype=torch.bfloat16)")


def _check_params(params):
    for p in params:
        _check_param_dtype(p)
        if not p.is_cuda:
            raise _lib.SpxError("libspx_hip works on HIP device tensors only (got a CPU parameter)")


_CAST_PARTS = 8  # matrices of one launch


def _in_one_launch(params) -> bool:
    return len(params) <= _CAST_PARTS and all(
        p.is_cuda and p.is_contiguous() and p.numel() % 8 == 0 and p.numel() > 0 and p.data_ptr() % 16 == 0
        and p.dtype in (torch.float32, torch.bfloat16) for p in params)


def _cast_together(groups):
    """The bf16 copies of several fp32 weights, or merged weights, from one launch: views of one buffer, 256 bytes aligned
    as an allocation of their own would be -- or None, where they are not all fp32 parameters that one launch takes.
    (q k v, o, gate up, down of the 1B shape in a training pass: 97 us in four launches, 66 in one.)"""
    params = [p for g in groups for p in g]
    if (len(groups) < 2 or not _in_one_launch(params) or len({p.device for p in params}) > 1
            or not all(p.dtype == torch.float32 and p.dim() == 2 and p.requires_grad for p in params)
            or not all(p.shape[1] == g[0].shape[1] for g in groups for p in g)):
        return None
    sizes = [sum(p.numel() for p in g) for g in groups]
    if any(n % 128 for n in sizes):
        return None
    flat = _lib.native().cat_bf16(*(p.detach().view(-1) for p in params))
    return [w.view(-1, g[0].shape[1]) for w, g in zip(flat.split(sizes), groups, strict=True)]


def _cat_bf16(params) -> torch.Tensor:
    """Row-wise concatenation of the parameters as one bf16 tensor (one pass: the copies cast)."""
    if _in_one_launch(params):
        return _lib.native().cat_bf16(*params)
    if len(params) == 1:
        return params[0].detach().to(torch.bfloat16)
    rows = sum(p.shape[0] for p in params)
    out = torch.empty(rows, *params[0].shape[1:], device=params[0].device, dtype=torch.bfloat16)
    r = 0
    for p in params:
        out[r:r + p.shape[0]].copy_(p.detach())
        r += p.shape[0]
    return out


def _pair_as_it_lies(params) -> bool:
    """Whether products may read two parameters as the halves of one weight: bf16 matrices of one shape, whole and aligned, on one
    device."""
    if len(params) != 2:
        return False
    a, b = params
    return (a.dtype == b.dtype == torch.bfloat16 and a.dim() == 2 and a.shape == b.shape and a.shape[0] % 256 == 0
            and a.shape[1] % 64 == 0 and a.device == b.device and a.is_contiguous() and b.is_contiguous()
            and a.data_ptr() % 16 == 0 and b.data_ptr() % 16 == 0 and a.is_cuda)


def _as_it_lies(p: torch.Tensor) -> torch.Tensor:
    """A bf16 parameter used alone: itself -- or a copy in rows of aligned chunks where it is a matrix stored otherwise
    (column by column, at an odd address, with an odd or overlapping row stride): the GEMM kernels take none of these."""
    w = p.detach()
    if w.dim() == 2 and w.shape[1] % 8 == 0 and (w.stride(1) != 1 or w.stride(0) % 8 or w.stride(0) < w.shape[1]
                                                 or w.data_ptr() % 16):
        return w.clone(memory_format=torch.contiguous_format)
    return w


def transposed_copy(w: torch.Tensor) -> torch.Tensor:
    """``w.transpose(-1, -2)`` as a new contiguous tensor; a stack ``[E, N, K]`` is transposed
    matrix by matrix.  On the library's kernel where its alignment rules hold."""
    if (w.dtype == torch.bfloat16 and w.is_cuda and w.dim() in (2, 3) and w.is_contiguous()
            and w.shape[-1] % 8 == 0 and w.shape[-2] % 8 == 0 and w.data_ptr() % 16 == 0):
        r, c = w.shape[-2], w.shape[-1]
        batches = w.shape[0] if w.dim() == 3 else 1
        out = torch.empty(*w.shape[:-2], c, r, device=w.device, dtype=w.dtype)
        _lib.call("spx_transpose_bf16", w, c, r * c, out, r, r * c, r, c, batches,
                  _lib.stream_ptr(w.device))
        return out
    return w.transpose(-1, -2).contiguous()


def _tn_ok(t: torch.Tensor) -> bool:
    return (t.dtype == torch.bfloat16 and t.stride(1) == 1 and t.shape[1] % 8 == 0
            and t.stride(0) % 8 == 0 and t.data_ptr() % 16 == 0)


def wgrad_product(dy: torch.Tensor, x: torch.Tensor, acc: torch.Tensor | None) -> torch.Tensor:
    """``acc (+)= dy.T @ x`` with an fp32 result: on the transposing MFMA kernel of this library
    where its alignment rules hold, else on PyTorch's matmul."""
    if _tn_ok(dy) and _tn_ok(x):
        from .gemm import gemm_tn

        if acc is None:
            return gemm_tn(dy, x, out_dtype=torch.float32)
        return gemm_tn(dy, x, acc, accumulate=True)
    if acc is None:
        return torch.mm(dy.t(), x, out_dtype=torch.float32)
    return torch.addmm(acc, dy.t(), x, out_dtype=torch.float32, out=acc)


class _Uses:
    """The uses of one compute weight in a forward and its backward: the inputs they ran on and the output gradients that came
    back.  What the staging node holds -- not the ``Staged`` itself, whose token leads back to the node."""

    __slots__ = ("shape", "device", "uses", "trainable", "bf16_params", "applied", "_xs", "_fill", "_dys", "_live", "_extras",
                 "_marked", "_acc", "_task")

    def __init__(self, uses: int, bf16_params: bool):
        self.shape = self.device = None  # of the compute weight
        self.uses = uses
        self.trainable = False
        self.bf16_params = bf16_params  # the parameters are bf16: a gradient written once may be bf16 itself
        self.applied = 0   # products of this forward that add their gradient to _acc
        self._xs = None    # [uses * T, cols]: the inputs of the uses, one after the other
        self._fill = 0     # rows of _xs taken by products so far
        self._dys = None   # [uses * T, rows]: the output gradients, same row positions (backward only)
        self._live = []    # (first row, rows) of the uses whose backward has run
        self._extras = []  # (dy, x) of uses outside the buffers
        self._marked = False
        self._acc = None   # gradient buffer of uses that add their gradient themselves
        self._task = None     # the backward pass (autograd graph task) the recorded uses belong to

    # ---- forward side
    def x_slot(self, rows: int):
        """Where the input ``[rows, cols]`` of the next product against this weight should be
        written so that its weight gradient joins the one product over all uses; None when
        there is nothing to gain (frozen weight, no graph, a single use) or no room."""
        if not self.trainable or self.uses <= 1 or not torch.is_grad_enabled():
            return None
        if self._xs is None:
            self._xs = torch.empty(self.uses * rows, self.shape[1], device=self.device,
                                   dtype=torch.bfloat16)
        if self._fill + rows > self._xs.shape[0]:
            return None
        return self._xs[self._fill:self._fill + rows]

    def take(self, x2: torch.Tensor) -> int:
        """Called by a product's forward with its input: the first row of ``x2`` in the input
        buffer if it is the slot ``x_slot`` handed out (the slot is then taken), else -1."""
        xs = self._xs
        if xs is None:
            return -1
        rows = x2.shape[0]
        if (x2.data_ptr() == xs.data_ptr() + self._fill * xs.stride(0) * 2 and x2.is_contiguous()
                and x2.shape[1] == xs.shape[1] and self._fill + rows <= xs.shape[0]):
            self._fill += rows
            return self._fill - rows
        return -1

    # ---- backward side
    def drop(self):
        """Forgets what the uses recorded."""
        self._dys, self._live, self._extras, self._marked, self._acc = None, [], [], False, None

    def _enter_pass(self):
        """What the uses record belongs to ONE backward pass, which ends in ``finish`` when autograd
        reaches the staging node.  A pass that never got there (``autograd.grad`` for other inputs
        over a retained graph) must not leak its records into the next one."""
        task = torch._C._current_graph_task_id()
        if task != self._task:
            self.drop()
            self._task = task

    def dy_slot(self, r0: int, rows: int):
        """Where the output gradient of the use at rows ``r0`` belongs (None for a use outside the
        buffers): a backward that allocates its own result writes it here."""
        if r0 < 0:
            return None
        self._enter_pass()
        if self._dys is None:
            self._dys = torch.empty(self._xs.shape[0], self.shape[0], device=self.device,
                                    dtype=torch.bfloat16)
        return self._dys[r0:r0 + rows]

    def defer(self, r0: int, dy2: torch.Tensor, x2: torch.Tensor):
        """Record one use's ``(dy, x)`` for the weight-gradient product the staging node runs.
        Returns what the calling backward returns as the gradient of ``token``."""
        self._enter_pass()
        if r0 >= 0:
            slot = self.dy_slot(r0, dy2.shape[0])
            if dy2.data_ptr() != slot.data_ptr():
                slot.copy_(dy2)
            self._live.append((r0, dy2.shape[0]))
        else:
            self._extras.append((dy2, x2))
        return self.mark()

    def mark(self):
        """What a use's backward returns as the gradient of ``token``: the empty marker that makes
        autograd reach the staging node, once per backward; None afterwards."""
        self._enter_pass()
        if self._marked:
            return None
        self._marked = True
        return _lib.zero(self.device).expand(self.shape)

    def grad_buffer(self):
        """``(buffer, holds)``: the buffer of ``w``'s shape that uses which compute their weight
        gradient themselves (the grouped expert products) add it to, and whether an earlier use of
        this backward has written it already (the first one overwrites).  fp32 -- or bf16 when this is
        the forward's only use and the parameters are bf16: the same fp32 accumulation and the same one
        rounding as a cast of the fp32 buffer."""
        self._enter_pass()
        holds = self._acc is not None
        if not holds:
            once = self.bf16_params and self.applied == 1
            self._acc = torch.empty(self.shape, device=self.device,
                                    dtype=torch.bfloat16 if once else torch.float32)
        return self._acc, holds

    def sole(self):
        """``(dy, x)`` where one product is all there is to the weight gradient (the records are dropped then), else None."""
        self._enter_pass()  # (the node may be reached by other weights' uses alone)
        if self._acc is not None or len(self._extras) > 1 or bool(self._extras) == bool(self._live):
            return None
        if self._extras:
            pair = self._extras[0]
        else:
            live = sorted(self._live)
            if any(a + n != b for (a, n), (b, _) in zip(live, live[1:], strict=False)):
                return None
            rows = slice(live[0][0], live[-1][0] + live[-1][1])
            pair = self._dys[rows], self._xs[rows]
        if not (_tn_ok(pair[0]) and _tn_ok(pair[1])):
            return None
        self.drop()
        return pair

    def finish(self, bf16_ok: bool = False):
        """The fp32 weight gradient of every recorded use (None if there is none): one product
        per run of adjacent uses in the buffers -- normally one -- plus one per outside use.
        ``bf16_ok``: the parameters are bf16, so when ONE product is all there is, it writes bf16
        itself (the same fp32 accumulation and the same one rounding as a cast of its fp32 result)."""
        self._enter_pass()
        acc = self._acc
        runs: list = []
        for r0, n in sorted(self._live):
            if runs and runs[-1][0] + runs[-1][1] == r0:
                runs[-1][1] += n
            else:
                runs.append([r0, n])
        if bf16_ok and acc is None and len(runs) == 1 and not self._extras:
            r0, n = runs[0]
            dy, x = self._dys[r0:r0 + n], self._xs[r0:r0 + n]
            if _tn_ok(dy) and _tn_ok(x):
                from .gemm import gemm_tn

                self._dys, self._live, self._marked = None, [], False
                return gemm_tn(dy, x, out_dtype=torch.bfloat16)
        if bf16_ok and acc is None and not runs and len(self._extras) == 1:
            dy, x = self._extras[0]
            if _tn_ok(dy) and _tn_ok(x):
                from .gemm import gemm_tn

                self._extras, self._marked = [], False
                return gemm_tn(dy, x, out_dtype=torch.bfloat16)
        for r0, n in runs:
            acc = wgrad_product(self._dys[r0:r0 + n], self._xs[r0:r0 + n], acc)
        for dy2, x2 in self._extras:
            acc = wgrad_product(dy2, x2, acc)
        self.drop()
        return acc


class Staged:
    """One compute weight of this forward.  ``w``: bf16 ``[rows, cols]`` (or 1-D for a norm gain); where products may read its two
    bf16 parameters as they lie (``pieces``, ``gemm.pair_routes``) it is put together when it is first asked for.
    ``rows_of``: the row count of every parameter in it; ``uses``: how many products the forward is expected to run against
    it (the size of the input / output-gradient buffers)."""

    __slots__ = ("_w", "pieces", "token", "rows_of", "_wt", "records", "x_slot", "take", "dy_slot", "defer", "mark", "grad_buffer")

    def __init__(self, w, rows_of, uses: int = 1, bf16_params: bool = False):
        self._w, self.pieces = w if isinstance(w, tuple) else (w, None)
        self.token = None  # fp32 stand-in of w's shape that carries the gradient edge (trainable only)
        self.rows_of = rows_of
        self._wt = None
        r = self.records = _Uses(uses, bf16_params)
        self.x_slot, self.take = r.x_slot, r.take
        self.dy_slot, self.defer, self.mark, self.grad_buffer = r.dy_slot, r.defer, r.mark, r.grad_buffer

    def train(self, w, token):
        """The compute weight and its token, as the staging node made them."""
        self._w, self.pieces = w if isinstance(w, tuple) else (w, None)
        self.token = token
        r = self.records
        r.shape, r.device, r.trainable = token.shape, token.device, True

    @property
    def w(self) -> torch.Tensor:
        if self._w is None:
            self._w = _cat_bf16(self.pieces)
        return self._w

    @property
    def trainable(self) -> bool:
        return self.token is not None

    @property
    def uses(self) -> int:
        return self.records.uses

    @property
    def applied(self) -> int:
        return self.records.applied

    @applied.setter
    def applied(self, n: int):
        self.records.applied = n

    @property
    def has_wt(self) -> bool:
        return self._wt is not None

    @property
    def wt(self) -> torch.Tensor:
        """``w.T`` contiguous (made on first use, kept with the staged weight)."""
        if self._wt is None:
            self._wt = transposed_copy(self.w.detach())
        return self._wt


class _Stage(torch.autograd.Function):
    """params -> (their bf16 row-wise concatenation, the fp32 token that carries its gradient);
    backward: the weight-gradient product over all recorded uses (``_Uses.finish``), split and
    cast to each parameter's dtype."""

    @staticmethod
    def forward(ctx, records: _Uses, *params):
        ctx.records = records
        ctx.rows = [p.shape[0] for p in params]
        ctx.dtypes = [p.dtype for p in params]
        if len(params) == 1 and params[0].dtype == torch.bfloat16:
            w = _as_it_lies(params[0])
        else:
            w = _cat_bf16(params)
        token = _lib.zero(w.device).expand(w.shape)
        ctx.mark_non_differentiable(w)
        ctx.set_materialize_grads(False)
        return w, token

    @staticmethod
    def backward(ctx, _gw, g):
        # g is the marker of ``_Uses.defer`` (no memory behind it): the gradient is computed here,
        # now that every use has run its backward
        acc = ctx.records.finish(bf16_ok=all(dt == torch.bfloat16 for dt in ctx.dtypes))
        if acc is not None:
            g = acc
        if g is None:
            return (None,) * (1 + len(ctx.rows))
        return (None, *_param_grads(g, ctx.rows, ctx.dtypes, ctx.needs_input_grad[1:]))


def _param_grads(g, rows, dtypes, needed):
    """The gradients of the parameters that a compute weight with gradient ``g`` is made of."""
    parts = g.split(rows, dim=0) if len(rows) > 1 else (g,)
    # (a part of a merged buffer is copied where its dtype changes)
    return [part.to(dt) if need else None for part, dt, need in zip(parts, dtypes, needed, strict=True)]


class _StageAll(torch.autograd.Function):
    """``_Stage`` of several compute weights whose uses end together (the weights of a layer): their weight gradients are one
    launch where that is faster (``gemm.gemm_tn_all``)."""

    @staticmethod
    def forward(ctx, records, made, sizes, *params):
        ctx.records, ctx.sizes = records, sizes
        ctx.rows, ctx.dtypes = [p.shape[0] for p in params], [p.dtype for p in params]
        ctx.set_materialize_grads(False)
        out, at = [], 0
        for i, n in enumerate(sizes):
            group = params[at:at + n]
            at += n
            w = made.get(i)
            if w is None and _pair_as_it_lies(group):
                out += [None, _lib.zero(group[0].device).expand(2 * group[0].shape[0], group[0].shape[1])]
                continue
            if w is None:
                w = _as_it_lies(group[0]) if n == 1 and group[0].dtype == torch.bfloat16 else _cat_bf16(group)
            out += [w, _lib.zero(w.device).expand(w.shape)]
        ctx.mark_non_differentiable(*(w for w in out[::2] if w is not None))
        return tuple(out)

    @staticmethod
    def backward(ctx, *gs):
        from .gemm import gemm_tn_all

        # (a node a weight ran where its own weight was asked for: this one is reached where any of the layer's is)
        needed = _lib.native().wanted(ctx)
        groups, at = [], 0
        for n in ctx.sizes:
            groups.append(slice(at, at + n))
            at += n
        sums, together = [None] * len(groups), {torch.bfloat16: [], torch.float32: []}
        for i, (uses, group) in enumerate(zip(ctx.records, groups, strict=True)):
            g = gs[2 * i + 1]
            if not any(needed[group]):
                uses.drop()
                continue
            bf16 = all(dt == torch.bfloat16 for dt in ctx.dtypes[group])
            pair = uses.sole()
            if pair is not None:
                together[torch.bfloat16 if bf16 else torch.float32].append((i, pair))
            else:
                sums[i] = uses.finish(bf16_ok=bf16)
                if sums[i] is None:
                    sums[i] = g
        for dtype, members in together.items():
            if members:
                for (i, _), acc in zip(members, gemm_tn_all([pair for _, pair in members], dtype), strict=True):
                    sums[i] = acc
        grads = []
        for g, group in zip(sums, groups, strict=True):
            grads += [None] * (group.stop - group.start) if g is None else _param_grads(
                g, ctx.rows[group], ctx.dtypes[group], needed[group])
        return (None, None, None, *grads)


class _StageGains(torch.autograd.Function):
    """bf16 compute copies of RMSNorm gains (``1 + p`` for the zero-centred form).  Its backward
    adds what the uses left in each gain's ``GainGrads`` (reduced here, all of them in one launch) to whatever
    gradient arrives the ordinary way, in the parameter's dtype."""

    @staticmethod
    def forward(ctx, plus_one, grads, *ps):
        ctx.grads, ctx.dtypes = grads, [p.dtype for p in ps]
        ctx.set_materialize_grads(False)
        if plus_one:
            return tuple((1.0 + p.detach().float()).to(torch.bfloat16) for p in ps)
        out = [p.detach() if p.dtype == torch.bfloat16 else None for p in ps]
        cast = [i for i, w in enumerate(out) if w is None]
        for at in range(0, len(cast), 4):  # (four to a launch)
            some = cast[at:at + 4]
            joint = _cat_bf16([ps[i] for i in some])
            for i, w in zip(some, joint.split([ps[i].shape[0] for i in some]), strict=True):
                out[i] = w
        return tuple(out)

    @staticmethod
    def backward(ctx, *gs):
        taken = [grads.take() for grads in ctx.grads]
        # (where a gradient arrives the ordinary way too -- not just the empty marker -- the sum is formed in fp32)
        extra = [g if g is not None and (t is None or g.stride(0) != 0) else None for g, t in zip(gs, taken, strict=True)]
        args = []
        for t, g, dt in zip(taken, extra, ctx.dtypes, strict=True):
            if t is not None:
                args += [*t, int(g is not None or dt == torch.float32)]
        sums = iter(_lib.native().gain_sums(*args)) if args else iter(())
        out = []
        for t, g, dt in zip(taken, extra, ctx.dtypes, strict=True):
            total = g if t is None else next(sums)
            if t is not None and g is not None:
                total = total + g.float()
            out.append(None if total is None else total.to(dt))
        return (None, None, *out)


class WeightStager:
    """Hands out the ``Staged`` compute weights of one model.  ``begin()`` starts a forward."""

    def __init__(self):
        self._fwd: dict = {}
        self._frozen: dict = {}
        self._uses = 1

    def begin(self, uses: int = 1):
        """``uses``: how often the forward applies each trainable layer weight (the TTT / MTP
        step count)."""
        self._fwd = {}
        self._uses = max(int(uses), 1)

    def invalidate(self):
        """Forget every kept copy of a frozen weight (they are rebuilt on the next forward)."""
        self._frozen = {}
        self._fwd = {}

    def get_all(self, *groups):
        """``get`` of every group of parameters (None: None): those that train are staged by one node, and those that have to be
        cast are cast in one launch."""
        if torch.is_grad_enabled():
            new = {tuple(id(p) for p in g): g for g in groups if g is not None}
            new = [g for key, g in new.items() if key not in self._fwd]
            train = [g for g in new if any(p.requires_grad for p in g)]
            if len(train) > 1:
                self._stage_all(train, _cast_together(new) if _autocast_bf16(new[0][0].device.type) else None)
        return tuple(None if g is None else self.get(*g) for g in groups)

    def _stage_all(self, groups, made):
        """``made``: their bf16 copies where they are there already."""
        for g in groups:
            _check_params(g)
        staged = [Staged(None, [p.shape[0] for p in g], self._uses, all(p.dtype == torch.bfloat16 for p in g)) for g in groups]
        out = _StageAll.apply([st.records for st in staged], dict(enumerate(made or ())), [len(g) for g in groups],
                              *(p for g in groups for p in g))
        for st, g, w, token in zip(staged, groups, out[::2], out[1::2], strict=True):
            st.train((None, tuple(p.detach() for p in g)) if w is None else w, token)
            self._fwd[tuple(id(p) for p in g)] = st

    def get(self, *params) -> Staged:
        """The staged row-wise concatenation of ``params`` for the running forward."""
        key = tuple(id(p) for p in params)
        hit = self._fwd.get(key)
        if hit is not None:
            return hit
        _check_params(params)
        rows_of = [p.shape[0] for p in params]
        if torch.is_grad_enabled() and any(p.requires_grad for p in params):
            st = Staged(None, rows_of, self._uses, all(p.dtype == torch.bfloat16 for p in params))
            st.train(*_Stage.apply(st.records, *params))
        else:
            fkey = tuple((p.data_ptr(), p._version, p.dtype) for p in params)
            kept = self._frozen.get(key)
            if kept is None or kept[0] != fkey:
                if any(p.requires_grad for p in params) and _pair_as_it_lies(params):
                    w = None, tuple(p.detach() for p in params)
                else:
                    w = _as_it_lies(params[0]) if len(params) == 1 and params[0].dtype == torch.bfloat16 \
                        else _cat_bf16(params)
                kept = (fkey, Staged(w, rows_of, self._uses))
                if not any(p.requires_grad for p in params):
                    self._frozen[key] = kept  # trainable weights seen under no_grad are not kept
            st = kept[1]
        self._fwd[key] = st
        return st

    def gain(self, p: torch.Tensor, plus_one: bool = False) -> torch.Tensor:
        """A small 1-D weight (an RMSNorm gain) in bf16 for the running forward.  ``plus_one``: the
        gain is ``1 + p`` (evaluated in fp32), the form of the Qwen3-Next norms.  A trainable gain
        goes through an autograd node (``_StageGains``) and carries a ``fused_ops.GainGrads``: the
        norm kernels of all its uses leave their partial sums there, and the node reduces them
        once, after the last use's backward."""
        hit = self._fwd.get(("gain", id(p), plus_one))
        if hit is None:
            _check_param_dtype(p)
            if p.requires_grad and torch.is_grad_enabled():
                return self._stage_gains([p], plus_one)[0]
            if plus_one:
                hit = (1.0 + p.float()).to(torch.bfloat16)
            else:
                hit = p if p.dtype == torch.bfloat16 else p.to(torch.bfloat16)
            self._fwd["gain", id(p), plus_one] = hit
        return hit

    def gains(self, norms):
        """Stages the gains of these norms (modules with ``weight``) through one node where they train: one launch casts
        them (four at a time) and one sums their gradients, where each alone takes three launches.  The node runs when
        the last of their uses has run its backward: norms that belong together by that."""
        if not torch.is_grad_enabled():
            return
        ps = {id(n.weight): n.weight for n in norms if n.weight.requires_grad and n.weight.is_cuda
              and ("gain", id(n.weight), False) not in self._fwd}.values()
        autocast = _autocast_bf16()
        ps = [p for p in ps if p.dtype == torch.bfloat16 or (autocast and p.dtype == torch.float32)]
        if len(ps) > 1 and all(p.device == ps[0].device for p in ps):
            self._stage_gains(ps, False)

    def _stage_gains(self, ps, plus_one):
        from .fused_ops import GainGrads

        grads = [GainGrads() for _ in ps]
        out = _StageGains.apply(plus_one, grads, *ps)
        for p, w, g in zip(ps, out, grads, strict=True):
            w.spx_gain_grads = g
            self._fwd["gain", id(p), plus_one] = w
        return out
