"""A step's weighted sum of losses in one row pass behind the frozen head (spx_vocab_loss_terms_fwd_grad) against float64
on the same logits, at the vocabularies where the row pass can go wrong: the least it takes, a ragged last chunk, the most
its registers hold."""

import pytest
import torch

from speculators_amd import losses as L
from speculators_amd import metrics as MT

pytestmark = pytest.mark.gpu

TERMS = ['{"ce": 0.1, "tv": 0.9}', '{"tv": 1.5, "kl_div": 0.25}', '{"jsd": 1.0, "rkl": -0.5, "kl_div": 2.0, "tv": 0.0, "ce": 1.0}',
         "rkl", "jsd", "tv", '{"kl_div": 1.0, "ce": 0.5}']


def _term(name, x, y):
    """Row losses in float64."""
    lp, lt = x.log_softmax(-1), y.log_softmax(-1)
    p, t = lp.exp(), lt.exp()
    if name == "ce":
        return -lp.gather(-1, y.argmax(-1, keepdim=True)).squeeze(-1)
    if name == "kl_div":
        return (t * (lt - lp)).sum(-1)
    if name == "rkl":
        return (p * (lp - lt)).sum(-1)
    if name == "tv":
        return 1 - torch.minimum(p, t).sum(-1)
    lm = torch.log((p + t) / 2)
    return 0.5 * ((p * (lp - lm)).sum(-1) + (t * (lt - lm)).sum(-1))


def _inputs(t, vocab, seed=0, h=64):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(1, t, h, generator=g).bfloat16()
    w = (torch.randn(vocab, h, generator=g) * 0.35).bfloat16()
    y = (x[0].float() @ w.float().t() + torch.randn(t, vocab, generator=g)).bfloat16()
    y[0, 5] = y[0, vocab - 1] = 60.0  # a tie for the arg-max, nearly all of the mass
    mask = (torch.rand(1, t, generator=g) < 0.7).float()
    mask[0, 3:9] = 0
    mask[0, :3] = 1
    return x.cuda().requires_grad_(True), w.cuda(), y.unsqueeze(0).cuda(), mask.cuda()


def _steps(spec, x, w, y, mask, steps, targets=None, decay=0.8):
    prev = mask.bool().clone()
    total, cache, heads, ms = None, {}, [], {}
    for k in range(steps):
        head = MT.Head(x, w, w.t().contiguous())
        total, m, _ = MT.compute_metrics(head, y if targets is None else targets, mask, prev, k, decay,
                                         L.resolve_loss_config(spec), cache, total_in=total, return_pred=True)
        heads.append(head)
        ms.update(m)
    (dx,) = torch.autograd.grad(total * 3.0, x)
    return total.detach(), ms, dx, heads, prev


@pytest.mark.parametrize("vocab", [4096, 4104, 10008, 32768])
@pytest.mark.parametrize("spec", TERMS)
def test_terms_in_one_row_pass(spec, vocab):
    t, steps, decay = 33, 3, 0.8
    x, w, y, mask = _inputs(t, vocab)
    config = L.resolve_loss_config(spec)
    assert L.terms_fit(config, w, y, None, mask, t)
    total, ms, dx, heads, prev = _steps(spec, x, w, y, mask, steps)
    logits = heads[0].logits.detach().double().cpu()[0].requires_grad_(True)
    want = 0.0
    for k in range(steps):
        n = t - k
        yk, mk = y.double().cpu()[0, k:], mask.double().cpu()[0, k:]
        for name, (_, wt) in config.items():
            mean = decay ** k * (_term(name, logits[:n], yk) * mk).sum() / (mk.sum() + 1e-5)
            want = want + wt * mean
            if len(config) > 1:  # (fp32 sums over the vocabulary; differences of nearly equal probabilities)
                assert abs(ms[f"{name}_loss_{k}_sum"].item() - mean.item()) <= 2e-5 * max(abs(mean.item()), 1.0), (k, name)
    assert abs(total.item() - want.item()) <= 2e-5 * max(abs(want.item()), 1.0)
    (dl,) = torch.autograd.grad(want * 3.0, logits)
    ref = dl @ w.double().cpu()
    # the gradient rows are rounded to bf16 for the product and its result again: 2^-8 of the row each, doubled
    assert (dx[0].double().cpu() - ref).abs().max().item() <= 2 ** -6 * ref.abs().max().item()


@pytest.mark.parametrize("side", ["draft", "target", "both"])
def test_terms_where_columns_are_ruled_out(side):
    """jsd with columns at the type's lowest value: in the target, or in the draft by a head's row."""
    vocab = 4104
    x, w, y, mask = _inputs(33, vocab, seed=2)
    lowest = torch.finfo(torch.bfloat16).min
    if side != "target":
        x.data[..., 0] = 1.0
        w[::3], w[::3, 0] = 0.0, lowest
    if side != "draft":
        y[..., 1::3] = lowest
        if side == "both":
            y[..., ::6] = lowest
    total, _, dx, heads, _ = _steps("jsd", x, w, y, mask, 2)
    logits = heads[0].logits.detach().double().cpu()[0]
    assert side == "target" or bool((logits[:, ::3] < -3e38).all())
    want, dl = 0.0, torch.zeros_like(logits)
    for k in range(2):
        n = 33 - k
        lp, lt = logits[:n].log_softmax(-1), y.double().cpu()[0, k:].log_softmax(-1)
        lm = torch.logaddexp(lp, lt) - torch.tensor(2.0).double().log()
        p, t, mk = lp.exp(), lt.exp(), mask.double().cpu()[0, k:]
        a, b = torch.where(p > 0, lp - lm, 0.0), torch.where(t > 0, lt - lm, 0.0)
        wt = 0.8 ** k * mk / (mk.sum() + 1e-5)
        ext = (p * a).sum(-1)
        want = want + (wt * 0.5 * (ext + (t * b).sum(-1))).sum()
        dl[:n] += 3.0 * 0.5 * wt[:, None] * p * (a - ext[:, None])
    assert abs(total.item() - want.item()) <= 2e-5 * max(abs(want.item()), 1.0)
    keep = torch.ones(vocab, dtype=torch.bool)
    if side != "target":
        keep[::3] = False
        assert not bool(dl[:, ::3].any())
    ref = dl[:, keep] @ w.double().cpu()[keep]
    assert (dx[0].double().cpu() - ref).abs().max().item() <= 2 ** -6 * ref.abs().max().item()


@pytest.mark.parametrize("spec", TERMS)
def test_terms_count_and_chain_like_the_streaming_pass(spec, monkeypatch):
    got = []
    for one_pass in (True, False):
        monkeypatch.setattr(L, "HEAD_LOSS_ONE_PASS", one_pass)
        x, w, y, mask = _inputs(70, 8192, seed=3)
        got.append(_steps(spec, x, w, y, mask, 3))
    assert got[0][1].keys() == got[1][1].keys()
    for k, v in got[1][1].items():
        if "acc" in k or k.endswith("total"):
            assert torch.equal(got[0][1][k], v), k
        else:
            assert abs(got[0][1][k].item() - v.item()) <= 2e-5 * max(abs(v.item()), 1.0), k
    assert torch.equal(got[0][4], got[1][4])
    assert (got[0][2] - got[1][2]).abs().max() <= 2 ** -6 * got[1][2].abs().max()


@pytest.mark.parametrize("rows", [5, 300])
def test_terms_with_gathered_targets(rows):
    """Full-vocabulary targets read through d2t at the first step: the same as handing over the gathered rows, up to the
    order in which the target rows' statistics are summed."""
    vocab, vt = 4096, 9001
    x, w, y, mask = _inputs(rows, vocab, seed=5)
    g = torch.Generator().manual_seed(1)
    sel = torch.randperm(vt, generator=g)[:vocab].sort().values
    full = torch.randn(1, rows, vt, generator=g).bfloat16()
    full[0, :, sel] = y[0].cpu()
    gather = MT.TargetGather(full.cuda(), (sel - torch.arange(vocab)).cuda())
    a = _steps(TERMS[0], x, w, None, mask, 2, targets=gather)
    b = _steps(TERMS[0], x, w, y, mask, 2)
    assert torch.equal(gather.compact[0], y[0])
    assert abs(a[0].item() - b[0].item()) <= 1e-5 * abs(b[0].item())
    for k in b[1]:
        if "acc" in k:
            assert torch.equal(a[1][k], b[1][k]), k
    assert (a[2] - b[2]).abs().max() <= 2 ** -6 * b[2].abs().max()
