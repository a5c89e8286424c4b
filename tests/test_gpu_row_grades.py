"""The input gradient of a frozen head from unit-weight rows: the row weights go onto the product's fp32 sums
(spx_gemm_bf16_rows_graded), so that dx carries one rounding."""

import pytest
import torch

from speculators_amd import losses as L
from speculators_amd import metrics as MT

pytestmark = pytest.mark.gpu

SHAPES = [  # (tile, parts, M, N, K): the tiles of a product with a device row count, whole and in parts; 0: 256 x 256
    (3, 1, 300, 264, 1032), (3, 10, 96, 64, 4096), (1, 3, 513, 2048, 4096), (2, 1, 2500, 3080, 4104), (2, 2, 1300, 2048, 8192),
    (0, 4, 3001, 4096, 8200), (0, 1, 2100, 4096, 2048), (0, 1, 3001, 4091, 8200), (0, 1, 5000, 8192, 56)]


@pytest.mark.parametrize("tile,parts,m,n,k", SHAPES)
@pytest.mark.parametrize("live", [0, 1, 193, 10 ** 6])
def test_one_rounding_against_float64(tile, parts, m, n, k, live):
    from speculators_amd import _lib

    lib = _lib.load()
    assert lib.spx_gemm_auto_tile(2, m, n, k, 4) == tile
    g = torch.Generator(device="cuda").manual_seed(m + n)
    a = torch.randn(m, k, device="cuda", generator=g).bfloat16()
    b = torch.randn(n, k, device="cuda", generator=g).bfloat16()
    rows = min(live, m)
    row_of = torch.randperm(m + 9, device="cuda", generator=g).to(torch.int32)[:m].contiguous()
    weight = torch.rand(m + 9, device="cuda", generator=g) * 1e-3 + 1e-5
    scale, factor = torch.tensor(0.37, device="cuda"), 0.9
    by = (weight.double()[row_of[:rows].long()] * (scale.double() * factor)).unsqueeze(1)
    want = (a[:rows].double() @ b.double().t()) * by
    # half a unit in the last place of bf16 (eight bits: 2^-8 of the power of two below the value), and fp32 sums of k products
    # times a factor of three fp32 roundings
    bound = 2 ** -8 * torch.exp2(want.abs().clamp_min(1e-30).log2().floor())
    bound = bound + 2 ** -22 * (a[:rows].double().abs() @ b.double().abs().t()) * by
    got = []
    for pad in (0, 8):
        need = max(lib.spx_gemm_auto_workspace_bytes(2, m, n, k, 4) if tile else 0, parts * m * n * 4 if parts > 1 else 0)
        ws = torch.empty(need // 4, device="cuda") if need else None
        c = torch.full((m, n + pad), 2.0, dtype=torch.bfloat16, device="cuda")
        _lib.call("spx_gemm_bf16_rows_graded", a, k, b, k, c, n + pad, m, n, k,
                  torch.tensor([live], dtype=torch.int32, device="cuda"), row_of, weight, scale, factor, 4, parts if not tile else 4,
                  ws, need, _lib.stream_ptr(a.device))
        assert (c[:, n:] == 2).all() and (c[rows:] == 2).all()
        got.append(c[:rows, :n])
        assert rows == 0 or ((got[-1].double() - want).abs() <= bound).all()
    assert torch.equal(got[0], got[1])


def _unit(op, x, y):
    """Logits gradients for a row weight of one, in float64 (losses/fused.py:11-18)."""
    x = x.detach().double().requires_grad_(True)
    lp, lq = torch.log_softmax(x, -1), torch.log_softmax(y.double(), -1)
    if op == "kl_div":
        loss = (lq.exp() * (lq - lp)).sum()
    elif op == "ce":
        loss = -lp.gather(-1, y.argmax(-1, keepdim=True)).sum()
    elif op == "rkl":
        loss = (lp.exp() * (lp - lq)).sum()
    elif op == "jsd":
        lm = torch.logaddexp(lp, lq) - torch.log(torch.tensor(2.0, device=x.device).double())
        loss = 0.5 * ((lp.exp() * (lp - lm)).sum() + (lq.exp() * (lq - lm)).sum())
    else:
        loss = (1 - torch.minimum(lp.exp(), lq.exp()).sum(-1)).sum()
    return torch.autograd.grad(loss, x)[0]


@pytest.mark.parametrize("terms,blocks", [("kl_div", True), ("ce", True)] + [
    (terms, False) for terms in ("kl_div", "ce", "rkl", "jsd", "tv", '{"ce": 0.1, "tv": 0.9}')])
def test_head_gradient_carries_one_rounding(terms, blocks):
    """The relative error of dx (2-norm) behind the one-read row pass against that of a gradient whose logits part and result
    are rounded once each: two roundings of the result are 1.2 to 1.3 of it."""
    config = L.resolve_loss_config(terms)
    g = torch.Generator(device="cuda").manual_seed(7)
    t, h, vocab, bs = 96, 512, 4096, 8
    x = torch.randn(1, t, h, device="cuda", generator=g).bfloat16().requires_grad_(True)
    w = (torch.randn(vocab, h, device="cuda", generator=g) * 3 * h ** -0.5).bfloat16()
    y = (3 * torch.randn(1, t, vocab, device="cuda", generator=g)).bfloat16()
    mask = torch.rand(1, t, device="cuda", generator=g) * (torch.rand(1, t, device="cuda", generator=g) < 0.7)
    head = MT.Head(x, w, w.t().contiguous())
    if blocks:
        mask[:, ::bs] = 0
        loss, _ = MT.dflash_compute_metrics(head, y, mask, bs, 4.0, config)
        by = mask.double()[0] * MT.dflash_loss_decay(torch.arange(t, device="cuda") % bs, 4.0).double()
    else:
        loss, _ = MT.compute_metrics(head, y, mask, mask != 0, 0, 1.0, config)
        by = mask.double()[0]
    (dx,) = torch.autograd.grad(loss * 0.37, x)
    by = 0.37 * by / (mask.double().sum() + 1e-5)
    logits = (x.detach()[0].float() @ w.float().t()).bfloat16()
    unit = sum(weight * _unit(name, logits, y[0]) for name, (_, weight) in config.items())
    want = (unit @ w.double()) * by.unsqueeze(1)
    once = ((unit.bfloat16().double() @ w.double()) * by.unsqueeze(1)).bfloat16().double()
    assert (dx[0].double() - want).norm().item() <= 1.05 * (once - want).norm().item()
