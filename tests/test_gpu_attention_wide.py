"""Attention at head_dim 256 (``wide_pass`` of ``attn_fwd_kernel`` and ``attn_bwd_dq_kernel``, the latter at 64 too: the products of
a tile in one row with everything else spread beside them) against the explicit soft-max in float64 over the same rounded queries: odd row
counts around the 32-key halves, 64-key tiles and 128-row workgroups, rows and whole tiles a wave sees nothing of, and
scores whose maximum moves on in every half tile, in one jump, or never."""

import pytest
import torch

pytestmark = pytest.mark.gpu
LOG2E = 1.4426950408889634


def _reference(q, k, v, dense, scale, go):
    """``(out, dq, bound)`` by the float64 soft-max over bf16(q * scale * log2 e), which is what the kernels multiply with the
    keys.  ``bound``: what dq may be off by, element by element -- dS and dq are rounded to bf16 (2^-9 each, and twice that
    for the fp32 sums and the exponential of fp32 scores), and delta is taken with the rounded output."""
    q, k, v, dense, go = (x.cuda() for x in (q, k, v, dense, go))
    qs = (q.float() * (torch.tensor(scale, dtype=torch.float32) * LOG2E)).bfloat16().double()
    group = q.shape[1] // k.shape[1]
    kk, vv = (x.double().repeat_interleave(group, 1) for x in (k, v))
    p = torch.softmax((qs @ kk.transpose(-1, -2)).masked_fill(~dense, float("-inf")) * 0.6931471805599453, -1)
    out = p @ vv
    do = go.double().transpose(1, 2)
    ds = p * (do @ vv.transpose(-1, -2) - (do * out).sum(-1, keepdim=True))
    dq = scale * (ds @ kk)
    d_delta = 2.0 ** -8 * (do.abs() * out.abs()).sum(-1, keepdim=True)
    bound = scale * ((2.0 ** -7 * ds.abs() + d_delta * p) @ kk.abs()) + 2.0 ** -8 * dq.abs() + 1e-6
    return out.transpose(1, 2).cpu(), dq.cpu(), bound.cpu()


def _rows(t, hq, hkv, kind, d=256):
    g = torch.Generator().manual_seed(t + 7 * hq)
    q, k, v = (torch.randn(1, h, t, d, generator=g) for h in (hq, hkv, hkv))
    if kind != "flat":
        # a direction every query shares; the keys' share of it grows, falls, or jumps once: scores from 0 to about
        # +- 90 in steps the reference value has to follow (it is left alone up to a distance of 12 in the exponent of 2)
        u = torch.randn(d, generator=g)
        u /= u.norm()
        ramp = {"rise": torch.linspace(0., 1., t), "fall": torch.linspace(1., 0., t),
                "jump": (torch.arange(t) == 2 * t // 3).float()}[kind]
        q += 8 * u
        k += (ramp * 7.8 * d ** 0.5)[None, None, :, None] * u
    return tuple(x.bfloat16() for x in (q, k, v))


def _check(fn, q, k, v, mask, dense):
    scale = q.shape[3] ** -0.5
    go = torch.randn(1, q.shape[2], q.shape[1], q.shape[3], generator=torch.Generator().manual_seed(1)).bfloat16()
    qg = q.cuda().requires_grad_(True)
    out = fn(qg, k.cuda(), v.cuda(), mask, scale)
    out.backward(go.cuda())
    want, dq, bound = _reference(q, k, v, dense, scale, go)
    # bf16 probabilities and result: two roundings of 2^-9 of at most max |v|; the rest is fp32
    err = (out.detach().double().cpu() - want).abs().max().item()
    assert torch.isfinite(out).all() and err <= 2.0 ** -7 * v.float().abs().max().item(), err
    off = (qg.grad.double().cpu() - dq).abs()
    assert torch.isfinite(qg.grad).all() and (off <= bound).all(), ((off - bound).max().item(), off.max().item())


@pytest.mark.parametrize("d", [256, 64])
@pytest.mark.parametrize("kind", ["flat", "rise", "fall", "jump"])
@pytest.mark.parametrize("t,window,docs", [(1, None, 1), (31, None, 1), (33, None, 2), (64, None, 1), (97, 20, 1), (130, None, 3),
                                           (257, 40, 1), (333, None, 4), (1700, 100, 2), (1900, None, 1), (4977, None, 2)])
def test_rows_and_reference_moves(t, window, docs, kind, d):
    from oracle import masks as OMK
    from speculators_amd import attention as A

    hq, hkv = (64, 2) if t > 4000 else (8, 2) if t > 1000 else (4, 1)  # (from 1.56e9 scores on V comes out of a transposed copy)
    doc = torch.arange(t) * docs // t
    q, k, v = _rows(t, hq, hkv, kind, d)
    mask = A.create_ttt_mask(doc.cuda(), t, window)
    _check(A.ttt_attention, q, k, v, mask, OMK.ttt_mask_dense(doc, t, 0, window))


@pytest.mark.parametrize("d", [256, 64])
@pytest.mark.parametrize("kind", ["flat", "rise"])
@pytest.mark.parametrize("t,window", [(200, None), (777, 64)])
def test_two_intervals_per_row(t, window, kind, d):
    """Anchored blocks: context keys and the block's own keys are two passes over one accumulator."""
    from oracle import masks as OMK
    from speculators_amd import attention as A

    anchors = torch.arange(0, t - 1, 13)
    nq = 8 * len(anchors)
    doc = (torch.arange(t) > t // 3).long()
    q, _, _ = _rows(nq, 4, 2, kind, d)
    _, k, v = _rows(t + nq, 4, 2, kind, d)
    mask = A.create_dflash_mask(doc.cuda(), t, anchors.cuda(), 8, window)
    _check(A.dflash_attention, q, k, v, mask, OMK.dflash_mask_dense(doc, t, anchors, 8, window))
