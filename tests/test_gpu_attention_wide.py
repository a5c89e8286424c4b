"""Attention at head_dim 256 (``attn_fwd_kernel``'s ``wide_pass``: 64 products in a row with the soft-max of each half tile spread
beside them) against the explicit soft-max in float64 over the same rounded queries: odd row counts around the 32-key
halves, 64-key tiles and 128-row workgroups, rows and whole tiles a wave sees nothing of, and scores whose maximum
moves on in every half tile, in one jump, or never."""

import pytest
import torch

pytestmark = pytest.mark.gpu
LOG2E = 1.4426950408889634


def _reference(q, k, v, dense, scale):
    """float64 soft-max over bf16(q * scale * log2 e), which is what the kernel multiplies with the keys"""
    q, k, v, dense = (x.cuda() for x in (q, k, v, dense))
    qs = (q.float() * (torch.tensor(scale, dtype=torch.float32) * LOG2E)).bfloat16().double()
    group = q.shape[1] // k.shape[1]
    kk, vv = (x.double().repeat_interleave(group, 1) for x in (k, v))
    s = (qs @ kk.transpose(-1, -2)).masked_fill(~dense, float("-inf"))
    return (torch.softmax(s * 0.6931471805599453, -1) @ vv).transpose(1, 2).cpu()


def _rows(t, hq, hkv, kind, steps=1):
    g = torch.Generator().manual_seed(t + 7 * hq)
    q, k, v = (torch.randn(1, h, n, 256, generator=g) for h, n in ((hq, t), (hkv, steps * t), (hkv, steps * t)))
    if kind != "flat":
        # a direction every query shares; the keys' share of it grows, falls, or jumps once: scores from 0 to about
        # +- 90 in steps the reference value has to follow (it is left alone up to a distance of 12 in the exponent of 2)
        u = torch.randn(256, generator=g)
        u /= u.norm()
        n = steps * t
        ramp = {"rise": torch.linspace(0., 1., n), "fall": torch.linspace(1., 0., n),
                "jump": (torch.arange(n) == 2 * n // 3).float()}[kind]
        q += 8 * u
        k += (ramp * 125)[None, None, :, None] * u
    return tuple(x.bfloat16() for x in (q, k, v))


def _check(out, want, v):
    # bf16 probabilities and result: two roundings of 2^-9 of at most max |v|; the rest is fp32
    err = (out.double().cpu() - want).abs().max().item()
    assert torch.isfinite(out).all() and err <= 2.0 ** -7 * v.float().abs().max().item(), err


@pytest.mark.parametrize("kind", ["flat", "rise", "fall", "jump"])
@pytest.mark.parametrize("t,window,docs", [(1, None, 1), (31, None, 1), (33, None, 2), (64, None, 1), (97, 20, 1), (130, None, 3),
                                           (257, 40, 1), (333, None, 4), (1700, 100, 2), (1900, None, 1), (4977, None, 2)])
def test_rows_and_reference_moves(t, window, docs, kind):
    from oracle import masks as OMK
    from speculators_amd import attention as A

    hq, hkv = (64, 2) if t > 4000 else (8, 2) if t > 1000 else (4, 1)  # (from 1.56e9 scores on V comes out of a transposed copy)
    doc = torch.arange(t) * docs // t
    q, k, v = _rows(t, hq, hkv, kind)
    mask = A.create_ttt_mask(doc.cuda(), t, window)
    out = A.ttt_attention(q.cuda(), k.cuda(), v.cuda(), mask, 256 ** -0.5)
    _check(out, _reference(q, k, v, OMK.ttt_mask_dense(doc, t, 0, window), 256 ** -0.5), v)


@pytest.mark.parametrize("kind", ["flat", "rise"])
@pytest.mark.parametrize("t,window", [(200, None), (777, 64)])
def test_two_intervals_per_row(t, window, kind):
    """Anchored blocks: context keys and the block's own keys are two passes over one accumulator."""
    from oracle import masks as OMK
    from speculators_amd import attention as A

    anchors = torch.arange(0, t - 1, 13)
    nq = 8 * len(anchors)
    doc = (torch.arange(t) > t // 3).long()
    q, _, _ = _rows(nq, 4, 2, kind)
    _, k, v = _rows(t + nq, 4, 2, kind)
    mask = A.create_dflash_mask(doc.cuda(), t, anchors.cuda(), 8, window)
    out = A.dflash_attention(q.cuda(), k.cuda(), v.cuda(), mask, 256 ** -0.5)
    _check(out, _reference(q, k, v, OMK.dflash_mask_dense(doc, t, anchors, 8, window), 256 ** -0.5), v)
