"""bf16 Linear products on the MFMA GEMM kernel.

``linear(x, weight)`` is ``torch.nn.functional.linear`` without bias
(``x @ weight.T``) for bf16 tensors.  The backward computes the input gradient on the weight
as it lies (NN form), or with the NT kernel against a transposed copy of it
(``weight_t``, ``[K, N]`` contiguous) -- kept by the caller for frozen weights
such as ``lm_head`` (model.py:70-71) so it is made once.  The weight gradient is the
transposed-operand product ``gemm_tn``.
The models call the ``*_staged`` forms below with the compute weights of ``weights.WeightStager``.
"""

from __future__ import annotations

import ctypes
import functools
import os
import threading

import torch

from . import _lib
from . import fused_ops as FO

_MAX_SPAN = 0x7ffffff0 - 64  # bytes an operand of the weight-gradient product (gemm_tn) may span per call


_CUS = 256  # workgroups the chip runs at a time (one per compute unit for the GEMM kernels)

# parts the contraction of a live-rows product may be cut into (gemm_nt(split=True)); 1 = never cut
SPLIT_PARTS = int(os.environ.get("SPX_GEMM_SPLIT_PARTS", "4"))
if not 1 <= SPLIT_PARTS <= 8:
    raise ValueError(f"SPX_GEMM_SPLIT_PARTS must be 1 .. 8, got {SPLIT_PARTS}")


# parts the last round's tiles of such a product with graded rows may be cut into; where SPX_GEMM_SPLIT_PARTS is set, it bounds
# these, too
LIVE_TAIL_PARTS = SPLIT_PARTS if "SPX_GEMM_SPLIT_PARTS" in os.environ else 8
# parts the tiles of a mostly empty last round of a product may be cut into (spx_gemm_bf16_nt_tail); 1 = never
TAIL_PARTS = int(os.environ.get("SPX_GEMM_TAIL_PARTS", "4"))
if not 1 <= TAIL_PARTS <= 8:
    raise ValueError(f"SPX_GEMM_TAIL_PARTS must be 1 .. 8, got {TAIL_PARTS}")

class _Workspaces(threading.local):
    """One thread's buffers, by (device, stream); they go with the thread."""

    def __init__(self):
        self.held: dict = {}


_workspaces = _Workspaces()


def _split_workspace(device, numel: int) -> torch.Tensor:
    """The fp32 partials of a product cut along its contraction: one buffer per (thread, device, stream), kept
    and grown on demand, so a TTT loop does not allocate hundreds of MB per step for a workspace the
    kernel leaves untouched whenever the device-side row count asks for one part.  The launches of one thread
    on one stream are ordered, so consecutive products may share it; another thread's may come between the launches of a
    product."""
    held = _workspaces.held
    key = (device.index, _lib.stream_ptr(device))
    ws = held.get(key)
    if ws is None or ws.numel() < numel:
        ws = held[key] = torch.empty(numel, device=device, dtype=torch.float32)
    return ws


def gemm_nt(a: torch.Tensor, b: torch.Tensor, out: torch.Tensor | None = None,
            m_live: torch.Tensor | None = None, split: bool = False) -> torch.Tensor:
    """``a[M, K] @ b[N, K].T -> [M, N]`` (bf16, fp32 accumulation).

    ``m_live`` (a one-element int32 device tensor) says how many leading rows of ``a`` count:
    the rows from there on are neither read nor written, and the host never learns the
    number (no synchronisation).  ``split``: the kernel may cut the contraction into up to
    ``SPLIT_PARTS`` parts when the tiles of the rows that count would leave compute units idle
    (decided on the device from the row count; fp32 partials in a workspace, added in a fixed
    order)."""
    if a.dtype != torch.bfloat16 or b.dtype != torch.bfloat16:
        raise _lib.SpxError("gemm_nt takes bf16 operands")
    if a.dim() != 2 or b.dim() != 2 or a.shape[1] != b.shape[1]:
        raise ValueError(f"shape mismatch: a {tuple(a.shape)} b {tuple(b.shape)}")
    if a.stride(1) != 1:
        a = a.contiguous()
    if b.stride(1) != 1:
        b = b.contiguous()
    m, k = a.shape
    n = b.shape[0]
    if out is None:
        out = torch.empty(m, n, device=a.device, dtype=torch.bfloat16)
    # (operands of any size go in one launch: the kernel's 32-bit offsets are relative to a tile)
    st = _lib.stream_ptr(a.device)
    if m_live is None:
        # a last round of tiles that fills at most half the chip is cut along the contraction
        # (the kernel decides from the same numbers; here only whether the workspace is handed over)
        rem = (-(-m // 256) * -(-n // 256)) % _CUS
        if TAIL_PARTS > 1 and 0 < rem <= _CUS // 2 and k >= 64 * 16 * 2 and a.is_cuda:
            nbytes = _lib.native().spx_gemm_tail_workspace_bytes()
            ws = _split_workspace(a.device, nbytes // 4)
            _lib.call("spx_gemm_bf16_nt_tail", a, a.stride(0), b, b.stride(0),
                      out, out.stride(0), m, n, k, TAIL_PARTS, ws, nbytes, st)
            return out
        _lib.call("spx_gemm_bf16_nt", a, a.stride(0), b, b.stride(0),
                  out, out.stride(0), m, n, k, st)
    else:
        if m_live.dtype != torch.int32 or m_live.numel() != 1 or m_live.device != a.device:
            raise ValueError("m_live must be a one-element int32 tensor on the operands' device")
        # (a product of many rounds of tiles has little to gain from cutting: at most 1 / rounds)
        few_tiles = -(-m // 256) * -(-n // 256) <= 2 * 256
        if split and SPLIT_PARTS > 1 and few_tiles and n % 8 == 0 and out.stride(0) % 8 == 0 and k >= 64 * 16 * 2:
            ws = _split_workspace(a.device, SPLIT_PARTS * m * n)
            _lib.call("spx_gemm_bf16_nt_rows_split", a, a.stride(0), b, b.stride(0),
                      out, out.stride(0), m, n, k, m_live, SPLIT_PARTS, ws,
                      SPLIT_PARTS * m * n * 4, st)
        else:
            _lib.call("spx_gemm_bf16_nt_rows", a, a.stride(0), b, b.stride(0),
                      out, out.stride(0), m, n, k, m_live, st)
    return out


@functools.lru_cache(maxsize=4096)
def _plan(form: int, m: int, n: int, k: int, parts: int):
    """``(on the 256 x 256 kernel, workspace elements, predicted us)`` of ``spx_gemm_bf16_auto``."""
    lib = _lib.load()
    return (lib.spx_gemm_auto_tile(form, m, n, k, parts) == 0,
            lib.spx_gemm_auto_workspace_bytes(form, m, n, k, parts) // 4,
            lib.spx_gemm_auto_us(form, m, n, k, parts))


@functools.lru_cache(maxsize=4096)
def _graded_workspace(m: int, n: int, k: int, parts: int, split: int) -> int:
    """Workspace elements of ``spx_gemm_bf16_rows_graded``: all that it can use for any number of rows that count, up to 0.5 GB.
    (x 151936 -> 2048, room for 1280 partial tiles / so: 216 tiles in the last round whole 3592 us, in 7 parts 3438, 224 whole
    3625, in 8 parts 3507; behind a whole round 7210 / 7016 and 7213 / 7078; x 128256, 216 tiles 3055 / 2940.)"""
    return _lib.load().spx_gemm_graded_workspace_bytes(m, n, k, parts, split) // 4


# how a product runs, as csrc/layer_host.cpp numbers it: on spx_gemm_bf16_auto (NT or NN form), on the 256 x 256 kernel
# without or with its last round cut, or in the library
AUTO_NT, AUTO_NN, NT, TAIL, LINEAR, MATMUL, PAIR_NN, GATED_NT = range(8)


def _auto(form: int, a, b, ws_numel: int, m_live=None):
    ws = _split_workspace(a.device, ws_numel) if ws_numel else None
    return _lib.native().product(form, a, b, m_live, TAIL_PARTS, ws)


def matmul_nt(a: torch.Tensor, b: torch.Tensor, m_live: torch.Tensor | None = None) -> torch.Tensor:
    """``a[M, K] @ b[N, K].T`` (bf16) on the kernel its size asks for (``spx_gemm_bf16_auto``): products of
    few 256 x 256 tiles on smaller tiles or with the contraction in parts, the others on ``gemm_nt``.
    ``m_live`` as there (the 256 x 256 kernel then decides its parts from the row count)."""
    m, k = a.shape
    n = b.shape[0]
    if m_live is not None and (m_live.dtype != torch.int32 or m_live.numel() != 1 or m_live.device != a.device):
        raise ValueError("m_live must be a one-element int32 tensor on the operands' device")
    if k == b.shape[1] and k % 8 == 0 and a.stride(1) == 1 and b.stride(1) == 1 and a.dtype == b.dtype == torch.bfloat16:
        big, ws_numel, _ = _plan(0 if m_live is None else 2, m, n, k, TAIL_PARTS)
        if not big:
            return _auto(AUTO_NT, a, b, ws_numel, m_live)
    return gemm_nt(a, b, m_live=m_live, split=m_live is not None)


def rows_graded(a: torch.Tensor, b: torch.Tensor, m_live: torch.Tensor, row_of: torch.Tensor, row_weight: torch.Tensor,
                scale: torch.Tensor, factor: float) -> torch.Tensor:
    """``matmul_nt(a, b, m_live)`` with row ``m`` multiplied by ``row_weight[row_of[m]] * (scale * factor)`` in fp32, before its
    one rounding (``spx_gemm_bf16_rows_graded``).  The parts that are chosen on the device, and with them the order of the fp32
    sums, follow from the sizes and the row count alone, whatever product the workspace served before."""
    m, k = a.shape
    n = b.shape[0]
    if k != b.shape[1] or m_live.dtype != torch.int32 or row_of.dtype != torch.int32 or row_of.numel() < m:
        raise ValueError(f"a {tuple(a.shape)}, b {tuple(b.shape)}, int32 row count and rows")
    if row_weight.dtype != torch.float32 or scale.dtype != torch.float32 or not row_weight.is_contiguous():
        raise ValueError("row weights and scale are contiguous fp32")
    if b.stride(1) != 1:
        b = b.contiguous()
    parts = LIVE_TAIL_PARTS if SPLIT_PARTS > 1 else 1
    ws_numel = _graded_workspace(m, n, k, TAIL_PARTS, parts)
    ws = _split_workspace(a.device, ws_numel) if ws_numel else None
    out = torch.empty(m, n, device=a.device, dtype=torch.bfloat16)
    _lib.call("spx_gemm_bf16_rows_graded", a, a.stride(0), b, b.stride(0), out, n, m, n, k, m_live, row_of, row_weight, scale,
              factor, TAIL_PARTS, parts, ws, ws_numel * 4, _lib.stream_ptr(a.device))  # (the buffer may be larger: see above)
    return out


def _nn_fits(a: torch.Tensor, b: torch.Tensor) -> bool:
    """Whether ``a[M, K] @ b[K, N]`` meets the alignment rules of the NN kernels."""
    k, n = b.shape
    return (a.dtype == b.dtype == torch.bfloat16 and k % 8 == 0 and n % 8 == 0 and a.stride(1) == 1
            and b.stride(1) == 1 and a.stride(0) % 8 == 0 and b.stride(0) % 8 == 0 and a.data_ptr() % 16 == 0
            and b.data_ptr() % 16 == 0 and (k + 256) * b.stride(0) * 2 < _MAX_SPAN
            and (256 * a.stride(0) + k) * 2 < _MAX_SPAN)


def matmul_nn(a: torch.Tensor, b: torch.Tensor) -> torch.Tensor:
    """``a[M, K] @ b[K, N]`` (bf16, ``_nn_fits``): the input gradient of a Linear on its weight as it
    lies, no transposed copy of it."""
    m, k = a.shape
    n = b.shape[1]
    return _auto(AUTO_NN, a, b, _plan(1, m, n, k, TAIL_PARTS)[1])


# microseconds to transpose a million weight elements (spx_transpose_bf16: 4 bytes each at 3.8 TB/s)
_TRANSPOSE_US = 1.05


def input_gradient(dy2: torch.Tensor, staged) -> torch.Tensor:
    """``dy2 @ staged.w``: on the weight as it lies (NN kernels) or on its transposed copy (NT kernels), whichever
    is predicted to be faster -- the copy of a weight that trains is one per forward and is shared by the
    weight's uses; that of a frozen weight is kept."""
    if _nn_fits(dy2, staged.w):
        m, (k, n) = dy2.shape[0], staged.w.shape
        copy_us = 0.0 if staged.has_wt or not staged.trainable else _copy_us(k, n, staged.uses)
        if _plan(1, m, n, k, TAIL_PARTS)[2] <= _plan(0, m, n, k, TAIL_PARTS)[2] + copy_us:
            return matmul_nn(dy2, staged.w)
    return matmul_nt(dy2, staged.wt)


def gemm_nt_stats(a: torch.Tensor, b: torch.Tensor, store: bool = True, want_argmax: bool = True,
                  want_lse: bool = True):
    """``gemm_nt(a, b)`` whose epilogue also reduces every row of the (bf16-rounded) product to its
    soft-max statistics: returns ``(c [M, N] bf16 or None, lse [M] f32, argmax [M] i32 or None)``.
    ``store=False``: the product is not written at all (``c`` is None) -- the statistics are all a
    cross-entropy against arg-max targets needs of the verifier's logits."""
    if a.dtype != torch.bfloat16 or b.dtype != torch.bfloat16:
        raise _lib.SpxError("gemm_nt_stats takes bf16 operands")
    if a.dim() != 2 or b.dim() != 2 or a.shape[1] != b.shape[1]:
        raise ValueError(f"shape mismatch: a {tuple(a.shape)} b {tuple(b.shape)}")
    if a.stride(1) != 1:
        a = a.contiguous()
    if b.stride(1) != 1:
        b = b.contiguous()
    m, k = a.shape
    n = b.shape[0]
    dev = a.device
    out = torch.empty(m, n, device=dev, dtype=torch.bfloat16) if store else None
    if not (want_lse or want_argmax):
        raise ValueError("gemm_nt_stats: ask for the log-sum-exp, the arg-max or both")
    lse = torch.empty(m, device=dev, dtype=torch.float32) if want_lse else None
    am = torch.empty(m, device=dev, dtype=torch.int32) if want_argmax else None
    nbytes = _lib.native().spx_gemm_stats_workspace_bytes(m, n)
    ws = torch.empty(nbytes // 4, device=dev, dtype=torch.float32)
    _lib.call("spx_gemm_bf16_nt_stats", a, a.stride(0), b, b.stride(0),
              out, out.stride(0) if store else 0, m, n, k, lse, am, ws,
              nbytes, _lib.stream_ptr(dev))
    return out, lse, am




@functools.lru_cache(maxsize=4096)
def _split_bands(t: int, m: int, n: int) -> int:
    """How many parts the contraction of a ``[t, m]^T [t, n]`` product is cut into (``spx_gemm_bf16_tn_auto``)."""
    return _lib.load().spx_gemm_tn_parts(m, n, t)


class _TnProduct(ctypes.Structure):  # spx_tn_product
    _fields_ = [("a", ctypes.c_void_p), ("lda", ctypes.c_int64), ("b", ctypes.c_void_p), ("ldb", ctypes.c_int64),
                ("c", ctypes.c_void_p), ("ldc", ctypes.c_int64), ("M", ctypes.c_int64), ("N", ctypes.c_int64),
                ("T", ctypes.c_int64)]


@functools.lru_cache(maxsize=4096)
def _tn_list_plan(shapes: tuple, fp32: bool):
    """``(predicted us, workspace elements)`` of ``spx_gemm_bf16_tn_list`` over products ``(T, M, N, lda, ldb, ldc)``; us is
    negative where it does not take them."""
    lib = _lib.load()
    items = (_TnProduct * len(shapes))(*(_TnProduct(0, lda, 0, ldb, 0, ldc, m, n, t) for t, m, n, lda, ldb, ldc in shapes))
    return (lib.spx_gemm_tn_list_us(items, len(shapes), int(fp32)),
            lib.spx_gemm_tn_list_workspace_bytes(items, len(shapes), int(fp32)) // 4)


@functools.lru_cache(maxsize=4096)
def _tn_alone(shape: tuple, fp32: bool):
    """``(predicted us, on the walking kernel)`` of one weight gradient.  The walking kernel in the place of the 256 x 256
    kernel, and in the place of smaller tiles where it is predicted to be faster -- bf16 results by 8 %: the prices of the
    smaller tiles know no type of result and lie 5 % above what bf16 ones take, 10 % below fp32 (12 % rms).  1164 products of 130
    to 9000 rows, results of 48 to 3000 large tiles: 0.953 of the time without the walking kernel, 1.008 of the better of the two;
    21 take more than 1.03 of that time, the worst 1.19."""
    t, m, n = shape[:3]
    lib = _lib.load()
    us, walks = lib.spx_gemm_tn_us(m, n, t), _tn_list_plan((shape,), fp32)[0]
    taken = 0 < walks < us * (1.0 if fp32 else 0.92) or (walks > 0 and lib.spx_gemm_tn_tile(m, n, t) == 0)
    return (walks if taken else us), taken


def _tn_shape(a, b, out) -> tuple:
    n = b.shape[1]
    return a.shape[0], a.shape[1], n, a.stride(0), b.stride(0), n if out is None else out.stride(0)


def _walks(shape: tuple, fp32: bool) -> bool:
    return _tn_alone(shape, fp32)[1]


def _whole_lines(a, b, out) -> bool:
    return (a.data_ptr() % 16 == 0 and b.data_ptr() % 16 == 0 and a.shape[1] % 8 == 0 and b.shape[1] % 8 == 0
            and a.stride(0) % 8 == 0 and b.stride(0) % 8 == 0 and (out is None or out.data_ptr() % 16 == 0))


def _tn_list(pairs, fp32: bool, outs):
    ws_numel = _tn_list_plan(tuple(_tn_shape(a, b, out) for (a, b), out in zip(pairs, outs, strict=True)), fp32)[1]
    ws = _split_workspace(pairs[0][0].device, ws_numel) if ws_numel else None
    return _lib.native().products_tn(fp32, ws, *(x for (a, b), out in zip(pairs, outs, strict=True) for x in (a, b, out)))


def gemm_tn_all(pairs, out_dtype: torch.dtype):
    """``gemm_tn`` of every ``(a, b)``: in one launch where the walking kernel takes them all and is predicted to be faster than
    each alone (the layer of the 1B shape over 1536 rows: 219 us in four launches, 167 in one; prices of fp32 results
    as ``_tn_alone`` says.  457 lists of two to four products over 130 to 20000 rows: 0.76 of the time without the walking
    kernel, two above 1.03 of it, the worst 1.05; 1.004 of the better of one launch and several)."""
    fp32 = out_dtype == torch.float32
    shapes = tuple(_tn_shape(a, b, None) for a, b in pairs)
    if 1 < len(pairs) <= 8 and all(s[0] > 0 for s in shapes) and all(_whole_lines(a, b, None) for a, b in pairs):
        us = _tn_list_plan(shapes, fp32)[0]
        if 0 < us < sum(_tn_alone(s, fp32)[0] for s in shapes) * (1.08 if fp32 else 1.0):
            return _tn_list(pairs, fp32, [None] * len(pairs))
    return [gemm_tn(a, b, out_dtype=out_dtype) for a, b in pairs]


def gemm_tn(a: torch.Tensor, b: torch.Tensor, out: torch.Tensor | None = None,
            accumulate: bool = False, out_dtype: torch.dtype = torch.bfloat16) -> torch.Tensor:
    """``a[T, M].T @ b[T, N] -> [M, N]`` (bf16 operands, fp32 accumulation): the weight gradient
    ``dY.T @ X`` of a Linear.  ``accumulate`` adds the product to ``out``.  The result is bf16 or,
    with ``out_dtype=torch.float32`` (or an fp32 ``out``), fp32."""
    if a.dtype != torch.bfloat16 or b.dtype != torch.bfloat16:
        raise _lib.SpxError("gemm_tn takes bf16 operands")
    if a.dim() != 2 or b.dim() != 2 or a.shape[0] != b.shape[0]:
        raise ValueError(f"shape mismatch: a {tuple(a.shape)} b {tuple(b.shape)}")
    if a.stride(1) != 1:
        a = a.contiguous()
    if b.stride(1) != 1:
        b = b.contiguous()
    t, m = a.shape
    n = b.shape[1]
    if out is None:
        if accumulate:
            raise ValueError("accumulate needs the tensor to add to")
        if out_dtype not in (torch.bfloat16, torch.float32):
            raise ValueError("out_dtype must be bfloat16 or float32")
    elif out.shape != (m, n) or out.dtype not in (torch.bfloat16, torch.float32) or out.stride(1) != 1:
        raise ValueError(f"out must be a bf16 or fp32 [{m}, {n}] tensor with unit column stride")
    fp32 = (out_dtype if out is None else out.dtype) == torch.float32
    if not accumulate and t > 0 and _walks(_tn_shape(a, b, out), fp32) and _whole_lines(a, b, out):
        return _tn_list([(a, b)], fp32, [out])[0]
    # 32-bit byte offsets inside the kernel: a contraction that spans 2 GiB or more of an
    # operand is fed in bands of rows, every band after the first added to the result.  A bf16 result of several
    # bands is formed in fp32 and rounded once, like that of one
    rows = max(_MAX_SPAN // (2 * max(a.stride(0), b.stride(0))) - 256, 1)
    if t > rows and not fp32:
        total = gemm_tn(a, b, out.float() if accumulate else None, accumulate, torch.float32)
        return total.to(torch.bfloat16) if out is None else out.copy_(total)
    if t == 0:  # nothing to launch: the empty sum
        if out is None:
            return torch.zeros(m, n, device=a.device, dtype=out_dtype)
        return out if accumulate else out.zero_()
    for t0 in range(0, t, rows):
        # a small result with a long contraction: fp32 partials of its parts, summed in a fixed order
        parts = _split_bands(min(rows, t - t0), m, n)
        ws = _split_workspace(a.device, parts * m * n) if parts > 1 else None
        out = _lib.native().product_tn(a[t0:t0 + rows], b[t0:t0 + rows], out, accumulate or t0 > 0, fp32, ws)
    return out


class _Linear(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, weight, weight_t):
        x2 = x.reshape(-1, x.shape[-1])
        y = matmul_nt(x2, weight)
        ctx.save_for_backward(x2, weight, weight_t)
        ctx.x_shape = x.shape
        return y.view(*x.shape[:-1], weight.shape[0])

    @staticmethod
    def backward(ctx, dy):
        x2, weight, weight_t = ctx.saved_tensors
        dy2 = dy.reshape(-1, dy.shape[-1]).to(torch.bfloat16)
        dx = dw = None
        if ctx.needs_input_grad[0]:
            if weight_t is None and _nn_fits(dy2, weight):
                dx = matmul_nn(dy2, weight)
            else:
                dx = matmul_nt(dy2, weight_t if weight_t is not None else weight.t().contiguous())
            dx = dx.view(ctx.x_shape)
        if ctx.needs_input_grad[1]:
            from .weights import wgrad_product

            dw = wgrad_product(dy2 if dy2.stride(1) == 1 else dy2.contiguous(), x2, None).to(weight.dtype)
        return dx, dw, None


def linear(x: torch.Tensor, weight: torch.Tensor, weight_t: torch.Tensor | None = None):
    """``x[..., K] @ weight[N, K].T`` on the HIP GEMM; ``weight_t`` optionally holds
    ``weight.T`` contiguous for the backward."""
    return _Linear.apply(x, weight, weight_t)


# Which GEMM runs the decoder-layer projections (q/k/v, o, gate/up, down and their input
# gradients): "hipblaslt" = PyTorch's matmul (the library GEMM), "spx" = this library's MFMA kernels, "mixed" =
# each where it is faster: the forward products as ``_own_forward`` and ``_walking_forward`` say, the input gradients on
# this library's kernels (``input_gradient``: on the weight as it lies, or on its transposed copy).  The fc / lm_head /
# verifier-head products and every weight gradient always run on this library's kernels.
DECODER_GEMM = os.environ.get("SPX_DECODER_GEMM", "mixed")
if DECODER_GEMM not in ("hipblaslt", "spx", "mixed"):
    raise ValueError(f"SPX_DECODER_GEMM must be 'hipblaslt', 'spx' or 'mixed', got {DECODER_GEMM!r}")


@functools.lru_cache(maxsize=4096)
def _on_192_rows(m: int, n: int, k: int, parts: int) -> bool:
    """The part of ``_own_forward`` for products that the tiles of 192 rows took from whole rounds of the large ones."""
    tile = _lib.load().spx_gemm_auto_tile(0, m, n, k, parts)
    if tile == 5 and -(-m // 192) * -(-n // 192) <= 2 * _CUS:
        return True
    return tile in (4, 5) and m <= 1024 and k <= 3072


def _own_forward(m: int, n: int, k: int, parts: int | None = None) -> bool:
    """Whether the forward product of a decoder projection runs on this library's kernels in "mixed" (ratios: own time to
    hipBLASLt's).

    Chosen without the tiles of 192 rows: where smaller tiles fill the chip in one round (0.54 - 1.04 for 70 products of the
    1B, 8B and 70B shapes at 256 to 4096 rows, three 1.11 - 1.20), and where the last round of the large tiles is cut along
    the contraction (``spx_gemm_bf16_nt_tail``; 0.67 - 1.16 for 15, the merged q/k/v projection of the 8B shape at 4096 rows
    0.96).  What these choose may then run on tiles of 192 rows.

    Of the rest, whole rounds of the large tiles (mostly 1.01 - 1.13), what the tiles of 192 rows took: at most two rounds
    of 192 x 192 (29 products of 140 to 8199 rows 0.51 - 1.02, 0.81 in the geometric mean; 1B q/k/v at 2700 - 3072 rows 0.84 -
    0.91, 8B q/k/v at 1350 - 1536 0.92), and up to 1024 rows where the contraction is short: K to 3072 0.57 - 1.05 over 30
    products (0.83), from 4096 on 0.80 - 1.33 over 41 (1.06; 8B gate/up at 260 - 960 rows 0.99 - 1.11, 70B q/k/v at 777 - 1024
    1.24 - 1.33, 70B gate/up 1.02 - 1.21).
    (profiles/decoder_forward_products.txt.)"""
    parts = TAIL_PARTS if parts is None else parts
    big, ws_numel, _ = _plan(2, m, n, k, parts)  # (the choice without them is that of a device row count)
    if not big:
        if ws_numel > 0 or m <= 1024 or m * n <= 256 * 256 * 128:
            return True
    else:
        tiles = -(-m // 256) * -(-n // 256)
        if parts > 1 and 0 < tiles % _CUS <= _CUS // 2 and k >= 64 * 16 * 2 and tiles < 2 * _CUS:
            return True
    return _on_192_rows(m, n, k, parts)


def _walking_forward(m: int, n: int, k: int, parts: int | None = None) -> bool:
    """Of what ``_own_forward`` leaves to the library, the products that workgroups which walk the large tiles take as fast or
    faster (ratios: own time to hipBLASLt's, 156 products of 700 to 32760 rows of the 1B, 8B and 70B shapes and others; each is a
    library call of some 25 us on the host less, too).

    Contractions below 4096: 0.71 - 1.02 over 52 products, 0.95 in the geometric mean (1B gate/up 0.96 - 1.02, its results
    leave under the next tile's loads).  A last round cut along the contraction: 0.65 - 1.01 over 22 (0.86; 8B gate/up 0.77 -
    1.01, 70B gate/up 0.90 - 0.93).  Contractions from 16384 on: 0.64 - 1.02 over 22 (0.86).  Left to the library: whole
    rounds over 4096 to 16383, 0.84 - 1.05 over 55 (1.00, but 1.01 - 1.05 where N is a power of two or three of them), and
    the tiles of 192 rows."""
    return _walks_as_fast(m, n, k, TAIL_PARTS if parts is None else parts)


@functools.lru_cache(maxsize=4096)
def _walks_as_fast(m: int, n: int, k: int, parts: int) -> bool:
    if not m or k % 64 or k < 192 or n % 8 or _lib.load().spx_gemm_auto_tile(0, m, n, k, parts):
        return False
    if k < 4096:
        return True
    return m > 1024 and (k >= 16384 or _forward_route("spx", parts, m, n, k)[0] == TAIL)


def _rows_in_lines(t: torch.Tensor) -> bool:
    """Whether the 256 x 256 kernels read a matrix as it lies."""
    return t.stride(1) == 1 and t.stride(0) % 8 == 0 and t.shape[1] <= t.stride(0) < 1 << 21 and t.data_ptr() % 16 == 0


def _project(x2: torch.Tensor, staged) -> torch.Tensor:
    """``x2 @ staged.w.T`` of a decoder-layer projection."""
    if DECODER_GEMM == "spx":
        return matmul_nt(x2, staged.w)
    if DECODER_GEMM == "mixed" and x2.dtype == torch.bfloat16:
        m, (n, k) = x2.shape[0], staged.w.shape
        if _own_forward(m, n, k) or (_walking_forward(m, n, k) and _rows_in_lines(x2) and _rows_in_lines(staged.w)):
            return matmul_nt(x2, staged.w)
    return torch.nn.functional.linear(x2, staged.w)


def _project_back(dy2: torch.Tensor, staged) -> torch.Tensor:
    """``dy2 @ staged.w``: the input gradient of a decoder-layer projection."""
    # (the kernel contracts in chunks of 8: a projection a few columns wide -- a gate of width 1 --
    # stays with the library)
    if DECODER_GEMM != "hipblaslt" and dy2.shape[1] % 8 == 0 and dy2.stride(0) % 8 == 0 and dy2.stride(1) == 1:
        return input_gradient(dy2, staged)
    return torch.matmul(dy2, staged.w)


@functools.lru_cache(maxsize=4096)
def _lines_matter(mode: str, parts: int, m: int, n: int, k: int) -> bool:
    return mode == "mixed" and not _own_forward(m, n, k, parts) and _walking_forward(m, n, k, parts)


@functools.lru_cache(maxsize=4096)
def _forward_route(mode: str, parts: int, m: int, n: int, k: int, lines: bool = True):
    """``(route, workspace elements)`` of ``_project`` for contiguous rows (``lines``: of a weight of ``_rows_in_lines``)."""
    if mode == "hipblaslt" or (mode == "mixed" and not _own_forward(m, n, k, parts)
                               and not (lines and _walking_forward(m, n, k, parts))):
        return LINEAR, 0
    big, ws_numel, _ = _plan(0, m, n, k, parts)
    if not big and k % 8 == 0:
        return AUTO_NT, ws_numel
    rem = (-(-m // 256) * -(-n // 256)) % _CUS
    if parts > 1 and 0 < rem <= _CUS // 2 and k >= 64 * 16 * 2:
        return TAIL, _lib.native().spx_gemm_tail_workspace_bytes() // 4
    return NT, 0


def forward_route(m: int, staged):
    w = staged.w
    route = _forward_route(DECODER_GEMM, TAIL_PARTS, m, *w.shape)
    if _lines_matter(DECODER_GEMM, TAIL_PARTS, m, *w.shape) and not _rows_in_lines(w):
        return _forward_route(DECODER_GEMM, TAIL_PARTS, m, *w.shape, False)
    return route


@functools.lru_cache(maxsize=4096)
def _backward_route(mode: str, parts: int, m: int, k: int, n: int, ld: int, aligned: bool, copy_us: float):
    """``(route, workspace elements, on the transposed copy)`` of ``_project_back`` for contiguous rows."""
    if mode == "hipblaslt" or k % 8:
        return MATMUL, 0, False
    if aligned and n % 8 == 0 and ld % 8 == 0 and (k + 256) * ld * 2 < _MAX_SPAN and 257 * k * 2 < _MAX_SPAN:
        _, ws_numel, us = _plan(1, m, n, k, parts)
        if us <= _plan(0, m, n, k, parts)[2] + copy_us:
            return AUTO_NN, ws_numel, False
    return (*_forward_route("spx", parts, m, n, k), True)


def _copy_us(k: int, n: int, uses: int) -> float:
    """What the transposed copy of a weight costs each of its uses."""
    return (3.0 + _TRANSPOSE_US * 1e-6 * k * n) / uses


def backward_route(m: int, staged):
    """``(route, workspace elements, right operand)`` of the input gradient of a product with ``m`` rows."""
    w = staged.w
    k, n = w.shape
    copy_us = 0.0 if staged.has_wt or not staged.trainable else _copy_us(k, n, staged.uses)
    route, ws, transposed = _backward_route(DECODER_GEMM, TAIL_PARTS, m, k, n, w.stride(0), w.data_ptr() % 16 == 0,
                                            copy_us)
    return route, ws, staged.wt if transposed else w


@functools.lru_cache(maxsize=4096)
def _gated(mode: str, parts: int, m: int, f: int, h: int):
    """The workspace elements of the gated product, or None.  It is taken wherever its product would run on the large tiles here: against
    the product by its own route (the library's for a quarter of them) and the SwiGLU launch it took 0.61 - 1.02 of the time over 154 sizes
    of 15 widths (700 to 32760 rows, contractions of 896 to 8192) with the two results stored, 0.90 in the geometric mean, and 0.59 - 0.98
    without, 0.87."""
    if mode == "hipblaslt" or m <= 0 or not _lib.load().spx_gemm_gated_takes(m, f, h, h, parts):
        return None
    return _forward_route("spx", parts, m, 2 * f, h)[1]


def gated(m: int, staged, pair):
    """The workspace elements of the first product of an MLP with ``m`` rows where it forms its activation itself
    (``spx_gemm_bf16_gated``), else None; ``pair``: what ``pair_routes`` says."""
    w = staged.w if pair is None else staged.pieces[0]
    if w.stride(0) != w.shape[1] or w.data_ptr() % 16:
        return None
    return _gated(DECODER_GEMM, TAIL_PARTS, m, w.shape[0] // (2 if pair is None else 1), w.shape[1])


@functools.lru_cache(maxsize=4096)
def _pair_routes(mode: str, parts: int, m: int, f: int, h: int, trainable: bool, uses: int):
    """See ``pair_routes``.

    The concatenation that falls away reads and writes 4 f h bytes at 5 TB/s once a forward (8B shape 94 us, 1B 22 us; the products
    themselves take the same time, within 0.7 %: a validation pass of the 1B shape 1.013, the anchored-block draft of the 8B shape
    54.16 -> 53.97 ms).  The forward product is the gated one; the input gradient has to be one that is formed on the weight as it
    lies, by workgroups that walk the tiles."""
    if _gated(mode, parts, m, f, h) is None:
        return None
    if not trainable:
        return 0
    if not _lib.load().spx_gemm_pair_takes(1, m, h, 2 * f, h, parts) \
            or _plan(1, m, h, 2 * f, parts)[2] > _plan(0, m, h, 2 * f, parts)[2] + _copy_us(2 * f, h, uses):
        return None
    return _plan(1, m, h, 2 * f, parts)[1]


def pair_routes(m: int, staged):
    """Whether the products with ``m`` rows against a weight of two parameters take these as they lie (``spx_gemm_bf16_gated``,
    ``spx_gemm_bf16_pair``): the workspace elements of the input gradient, else None (they take ``staged.w``)."""
    if staged.pieces is None:
        return None
    return _pair_routes(DECODER_GEMM, TAIL_PARTS, m, *staged.pieces[0].shape, staged.trainable, staged.uses)


def workspace_for(device, *numels):
    """The workspace for products that ask for that many elements (one stream: they run one after the other)."""
    n = max(numels)
    return _split_workspace(device, n) if n else None


class _StagedLinear(torch.autograd.Function):
    """``x @ w.T`` against a staged weight (``weights.Staged``): on the MFMA kernel of this library
    (``hip``) or on PyTorch's hipBLASLt matmul.  The weight gradient is left to the staged weight,
    which computes it over all of its uses at once (``weights._Uses.defer``)."""

    @staticmethod
    def forward(ctx, x, _token, staged, hip: bool):
        if x.dtype != torch.bfloat16:
            raise _lib.SpxError("the HIP layer kernels take bf16 tensors")
        w = staged.w
        x2 = x.reshape(-1, x.shape[-1])
        y = matmul_nt(x2, w) if hip else _project(x2, staged)
        ctx.save_for_backward(x2, w)
        ctx.staged, ctx.hip, ctx.x_shape = staged, hip, x.shape
        ctx.slot = staged.take(x2) if ctx.needs_input_grad[1] else -1
        ctx.rows = x2.shape[0]
        return y.view(*x.shape[:-1], w.shape[0])

    @staticmethod
    def backward(ctx, dy):
        x2, w = ctx.saved_tensors
        dy2 = dy.reshape(-1, dy.shape[-1]).to(torch.bfloat16)
        dx = dw = None
        if ctx.needs_input_grad[0]:
            dx = (input_gradient(dy2, ctx.staged) if ctx.hip else _project_back(dy2, ctx.staged)).view(ctx.x_shape)
        if ctx.needs_input_grad[1]:
            dw = ctx.staged.defer(ctx.slot, dy2, x2)
        return dx, dw, None, None


def linear_staged(x: torch.Tensor, staged, hip: bool = False) -> torch.Tensor:
    """``x[..., K] @ staged.w[N, K].T``; see ``_StagedLinear``."""
    if not torch.is_grad_enabled() or not (x.requires_grad or staged.trainable):
        x2 = x.reshape(-1, x.shape[-1])
        y = matmul_nt(x2, staged.w) if hip else _project(x2, staged)
        return y.view(*x.shape[:-1], staged.w.shape[0])
    y = _StagedLinear.apply(x, staged.token, staged, hip)
    node = y.grad_fn
    if node is not None and getattr(node, "slot", -1) >= 0:
        # where the gradient of `y` belongs, for the backward that produces it (fused_ops._AddRMSNorm):
        # written there, it is not copied into the weight's output-gradient buffer afterwards
        y.spx_grad_slot = (staged, node.slot, node.rows)
    return y


def _qkv_heads(qkv, position_ids, inv_freq, hq: int, hkv: int, d: int, offset: int, scale: float, kv_out=None):
    """``qkv [T, (hq + 2 hkv) * d]`` -> rotated q and k, and v, head-major (``kv_out`` as in ``qkv_rope``)."""
    t, n = qkv.shape
    q = torch.empty(1, hq, t, d, device=qkv.device, dtype=torch.bfloat16)
    if kv_out is not None:
        # [1, Hkv, T, D] windows of the preallocated K / V cache: written in place
        k, v = kv_out
    else:
        kv = torch.empty(2, 1, hkv, t, d, device=qkv.device, dtype=torch.bfloat16)
        k, v = kv[0], kv[1]
    _lib.call("spx_rope_qkv", qkv, n, q, t * d, k, k.stride(1), v, v.stride(1), position_ids, inv_freq, t, hq, hkv, d,
              2 * inv_freq.numel(), 0, offset, scale, _lib.stream_ptr(qkv.device))
    return q, k, v


def _qkv_tokens(dqkv, grads, position_ids, inv_freq, hq: int, hkv: int, d: int, offset: int, scale: float):
    """The way back of ``_qkv_heads`` for the gradients ``grads`` (None: zeros) into ``dqkv``."""
    t, n = dqkv.shape
    dq, dk, dv = grads
    win = t * d
    _lib.call("spx_rope_qkv", dqkv, n, dq, dq.stride(1) if dq is not None else win,
              dk, dk.stride(1) if dk is not None else win, dv, dv.stride(1) if dv is not None else win, position_ids,
              inv_freq, t, hq, hkv, d, 2 * inv_freq.numel(), 1, offset, scale, _lib.stream_ptr(dqkv.device))


class _QKVRope(torch.autograd.Function):
    """q/k/v projections of one input as ONE GEMM against the staged concatenation of the three
    weights, followed by the rotary embedding + head-major relayout of each part.  The backward
    undoes the relayout into the three column blocks of one ``[T, Nq + 2 Nkv]`` buffer, so the
    input gradient is one GEMM (no per-projection partial results to add up); that buffer is the
    step's slot of the staged weight's output-gradient buffer, from which the weight gradient of
    all TTT steps comes as one product."""

    @staticmethod
    def forward(ctx, x, _token, staged, position_ids, inv_freq, hq, hkv, d, offset, kv_out=None):
        if x.dtype != torch.bfloat16:
            raise _lib.SpxError("the HIP layer kernels take bf16 tensors")
        wcat = staged.w
        t = x.shape[-2]
        x2 = x.reshape(t, x.shape[-1])
        qkv = _project(x2, staged)
        n = qkv.shape[1]
        scale = FO.table_scale_of(inv_freq)
        outs = _qkv_heads(qkv, position_ids, inv_freq, hq, hkv, d, offset, scale, kv_out)
        ctx.save_for_backward(x2, wcat, position_ids, inv_freq)
        ctx.meta = (x.shape, hq, hkv, d, offset, n, staged, scale)
        ctx.slot = staged.take(x2) if ctx.needs_input_grad[1] else -1
        ctx.set_materialize_grads(False)
        return outs

    @staticmethod
    def backward(ctx, dq, dk, dv):
        x2, wcat, position_ids, inv_freq = ctx.saved_tensors
        shape, hq, hkv, d, offset, n, staged, scale = ctx.meta
        t = x2.shape[0]
        dqkv = staged.dy_slot(ctx.slot, t) if ctx.needs_input_grad[1] else None
        if dqkv is None:
            dqkv = torch.empty(t, n, device=x2.device, dtype=torch.bfloat16)
        grads = []
        for g in (dq, dk, dv):
            if g is not None:
                g = g.to(torch.bfloat16)
                # a window of a longer gradient tensor is read in place through its head stride
                if not (g.stride(3) == 1 and g.stride(2) == d and g.stride(1) % 8 == 0
                        and g.stride(1) >= t * d and g.data_ptr() % 16 == 0):
                    g = g.contiguous()
            grads.append(g)
        _qkv_tokens(dqkv, grads, position_ids, inv_freq, hq, hkv, d, offset, scale)
        dx = dw = None
        if ctx.needs_input_grad[0]:
            dx = _project_back(dqkv, staged).view(shape)
        if ctx.needs_input_grad[1]:
            dw = staged.defer(ctx.slot, dqkv, x2)
        return (dx, dw) + (None,) * 8


def qkv_rope(x, staged, position_ids, inv_freq, hq: int, hkv: int, d: int, offset: int, kv_out=None):
    """``(q [1,Hq,T,D], k [1,Hkv,T,D], v [1,Hkv,T,D])`` with the rotary embedding at
    ``position_ids + offset`` applied to q and k; ``staged`` holds the row-wise concatenation of
    the q, k and v weights.  ``kv_out = (k_window, v_window)``: write k and v straight into these
    ``[1, Hkv, T, D]`` windows of a K / V cache and return them."""
    return _QKVRope.apply(x, staged.token, staged, position_ids, inv_freq, hq, hkv, d, offset, kv_out)


class _GateUpSwiGLU(torch.autograd.Function):
    """``silu(x @ Wg.T) * (x @ Wu.T)`` with the two projections as ONE GEMM against the staged
    concatenation of the two weights; the SwiGLU kernels read (and, in the backward, write) the two
    column halves of the merged ``[T, 2F]`` buffer in place, so the input gradient is one GEMM; the
    backward's ``[T, 2F]`` buffer is the step's slot of the staged weight's output-gradient buffer,
    from which the weight gradient of all TTT steps comes as one product.  ``out``: where the
    result goes (the input slot of the down projection's staged weight)."""

    @staticmethod
    def forward(ctx, x, _token, staged, out=None):
        if x.dtype != torch.bfloat16:
            raise _lib.SpxError("the HIP layer kernels take bf16 tensors")
        wcat = staged.w
        x2 = x.reshape(-1, x.shape[-1])
        f = wcat.shape[0] // 2
        gu = _project(x2, staged)  # [T, 2F]
        rows = x2.shape[0]
        if out is None or out.shape != (rows, f) or not out.is_contiguous():
            out = torch.empty(rows, f, device=x.device, dtype=torch.bfloat16)
        _lib.call("spx_swiglu_rows_fwd", gu, 2 * f, gu[:, f:], 2 * f, out, f,
                  rows, f, _lib.stream_ptr(x.device))
        ctx.save_for_backward(x2, gu, wcat)
        ctx.meta = (x.shape, f, staged)
        ctx.slot = staged.take(x2) if ctx.needs_input_grad[1] else -1
        return out.view(*x.shape[:-1], f)

    @staticmethod
    def backward(ctx, dout):
        x2, gu, wcat = ctx.saved_tensors
        shape, f, staged = ctx.meta
        rows = x2.shape[0]
        d2 = dout.reshape(rows, f).to(torch.bfloat16)
        if d2.stride(1) != 1 or d2.stride(0) % 8:
            d2 = d2.contiguous()
        dgu = staged.dy_slot(ctx.slot, rows) if ctx.needs_input_grad[1] else None
        if dgu is None:
            dgu = torch.empty(rows, 2 * f, device=x2.device, dtype=torch.bfloat16)
        _lib.call("spx_swiglu_rows_bwd", gu, 2 * f, gu[:, f:], 2 * f, d2,
                  d2.stride(0), dgu, 2 * f, dgu[:, f:], 2 * f, rows, f,
                  _lib.stream_ptr(x2.device))
        dx = dw = None
        if ctx.needs_input_grad[0]:
            dx = _project_back(dgu, staged).view(shape)
        if ctx.needs_input_grad[1]:
            dw = staged.defer(ctx.slot, dgu, x2)
        return dx, dw, None, None


def gate_up_swiglu(x, staged, out=None):
    """See ``_GateUpSwiGLU``; ``staged`` holds the row-wise concatenation of the gate and up
    weights."""
    return _GateUpSwiGLU.apply(x, staged.token, staged, out)
