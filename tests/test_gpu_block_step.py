"""The launches around an anchored-block step: its inputs (spx_dflash_inputs), the reduction that also leaves the metrics
(spx_block_total), and the one-read row pass behind the head with that reduction."""

import pytest
import torch

from speculators_amd import _lib
from speculators_amd import losses as L
from speculators_amd import metrics as MT
from speculators_amd.dflash import DFlashConfig, DFlashDraftModel

pytestmark = pytest.mark.gpu


def _model(bs, from_anchor):
    return DFlashDraftModel(DFlashConfig(hidden_size=64, num_attention_heads=1, num_key_value_heads=1, head_dim=64,
                                         intermediate_size=64, vocab_size=500, draft_vocab_size=64, num_aux=1,
                                         num_hidden_layers=1, block_size=bs, mask_token_id=499,
                                         sample_from_anchor=from_anchor))


@pytest.mark.parametrize("t,bs,anchors,valid", [(40, 5, [1, 7, 35, 0], [1, 1, 1, 0]), (257, 16, list(range(0, 240, 3)), None),
                                                (8, 8, [0], [1]), (300, 1, [299, -1, -300], None)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bool, torch.int64, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("from_anchor", [False, True])
def test_step_inputs(t, bs, anchors, valid, dtype, from_anchor):
    g = torch.Generator().manual_seed(t)
    ids, pos = torch.randint(0, 499, (1, t), generator=g), torch.randint(0, 1000, (1, t), generator=g)
    mask = (torch.rand(1, t, generator=g) < 0.6).to(dtype)
    a = torch.tensor(anchors)
    v = torch.ones(len(anchors), dtype=torch.bool) if valid is None else torch.tensor(valid).bool()
    out_ids, q_pos, kv_pos, idx, aligned = (x.cpu() for x in _model(bs, from_anchor)._inputs(
        ids.cuda(), pos.cuda(), mask.cuda(), a.cuda(), v.cuda(), t))
    rows = ((a % t)[:, None] + torch.arange(bs)).reshape(-1)
    want = torch.full((1, len(anchors) * bs), 499)
    want[:, ::bs] = ids[:, a]
    assert torch.equal(out_ids, want)
    block_pos = (pos[0, a][:, None] + torch.arange(bs)).reshape(-1)
    assert torch.equal(q_pos, block_pos) and torch.equal(kv_pos, torch.cat([pos[0], block_pos]))
    assert torch.equal(idx, rows if from_anchor else (rows - 1) % t)
    w = mask[:, rows].float() * v.repeat_interleave(bs)
    if not from_anchor:
        w[:, ::bs] = 0
    assert torch.equal(aligned, w)


def test_a_block_that_leaves_the_sequence_shows_in_the_mask():
    ids = torch.zeros(1, 20, dtype=torch.int64, device="cuda")
    mask = torch.ones(1, 20, device="cuda")
    for a, ok, bad in (([18], [True], 2), ([18], [False], 0), ([25], [True], 4), ([-30], [True], 4)):
        *_, aligned = _model(4, True)._inputs(ids, ids, mask, torch.tensor(a, device="cuda"),
                                              torch.tensor(ok, device="cuda"), 20)
        assert int(aligned.isnan().sum()) == bad, a


@pytest.mark.parametrize("bs,n", [(1, 5), (8, 24), (16, 4096), (5, 2005)])
@pytest.mark.parametrize("from_anchor", [False, True])
@pytest.mark.parametrize("weights", [False, True])
def test_block_total(bs, n, from_anchor, weights):
    g = torch.Generator().manual_seed(n)
    loss, mask = torch.rand(n, generator=g), (torch.rand(n, generator=g) < 0.7).float()
    am_d, am_t = (torch.randint(0, 3, (n,), generator=g, dtype=torch.int32) for _ in range(2))
    pw = torch.rand(n, generator=g) if weights else None
    gamma, factor, before = 4.0, 0.3, torch.tensor(2.5)
    dev = [x.cuda() if x is not None else None for x in (loss, am_d, am_t, mask, pw)]
    out = torch.full((9 + 2 * bs,), float("nan"), device="cuda")
    total, rw = torch.empty((), device="cuda"), torch.empty(n, device="cuda")
    _lib.call("spx_block_total", dev[0], dev[1], dev[2], dev[3], 3, dev[4], gamma, int(from_anchor), n, bs, factor,
              before.cuda(), total, out, rw, _lib.stream_ptr(out.device))
    slot = torch.arange(n) % bs
    w = pw.double() if weights else MT.dflash_loss_decay(slot.double(), gamma, from_anchor).double()
    want = mask.double() * w / (mask.double().sum() + 1e-5)
    mean = (loss.double() * want).sum()
    assert (rw.double().cpu() - want).abs().max() <= 1e-6 * want.abs().max() + 1e-12
    assert abs(out[0].item() - mean.item()) <= 2e-6 * max(mean.item(), 1e-3)
    assert abs(total.item() - (2.5 + factor * mean.item())) <= 1e-6 * 2.5 and out[2] == total
    hit = torch.stack([((am_d == am_t) & (mask != 0) & (slot == s)).sum() for s in range(bs)]).float()
    rows = torch.stack([((mask != 0) & (slot == s)).sum() for s in range(bs)]).float()
    assert torch.equal(out[9:9 + bs].cpu(), hit) and torch.equal(out[9 + bs:].cpu(), rows)
    first = 0 if from_anchor else 1
    eal = torch.cumprod(hit[first:].double() / rows[first:].double().clamp(min=1), 0).sum()
    assert out[3] == hit[first:].sum() and out[4] == rows[first:].sum()
    assert abs(out[5].item() - eal.item()) <= 1e-6 * max(eal.item(), 1.0)
    assert out[6:9].tolist() == [1.0] * 3


@pytest.mark.parametrize("vocab", [4096, 10008])
@pytest.mark.parametrize("loss_fn,weighting", [("kl_div", "fixed-exp-decay"), ("ce", "fixed-exp-decay"), ("kl_div", "dpace")])
def test_one_row_pass_against_the_streaming_form(vocab, loss_fn, weighting, monkeypatch):
    """Counts identical, loss within fp32 sums, the gradient within two bf16 roundings of its largest entry."""
    g = torch.Generator().manual_seed(vocab)
    n, bs, h = 96, 8, 64
    x0 = torch.randn(1, n, h, generator=g).bfloat16()
    w = (torch.randn(vocab, h, generator=g) * 0.35).bfloat16().cuda()
    y = torch.randn(1, n, vocab, generator=g).bfloat16().cuda()
    mask = (torch.rand(1, n, generator=g) < 0.7).float().cuda()
    mask[:, ::bs] = 0
    got = []
    for one_pass in (True, False):
        monkeypatch.setattr(L, "HEAD_LOSS_ONE_PASS", one_pass)
        x = x0.cuda().requires_grad_(True)
        loss, m = MT.dflash_compute_metrics(MT.Head(x, w, w.t().contiguous()), y, mask, bs, 4.0,
                                            L.resolve_loss_config(loss_fn), weighting)
        (dx,) = torch.autograd.grad(loss * 2.0, x)
        got.append((loss.detach(), m, dx))
    assert abs(got[0][0].item() - got[1][0].item()) <= 2e-6 * abs(got[1][0].item())
    for k, v in got[1][1].items():
        if "acc" in k or k.endswith("total") or k.startswith("eal"):
            assert torch.equal(got[0][1][k], v), k
    assert (got[0][2] - got[1][2]).abs().max() <= 2 ** -6 * got[1][2].abs().max()
    assert (got[0][2][0][mask[0] == 0] == 0).all()
