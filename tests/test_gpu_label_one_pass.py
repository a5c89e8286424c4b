"""The frozen-head cross-entropy whose row pass leaves the logits gradient behind, against the two-pass form and float64."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _case(rows, vocab, hidden, seed, live=0.7):
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn(rows, hidden, device="cuda", generator=g).bfloat16()
    w = (torch.randn(vocab, hidden, device="cuda", generator=g) * 0.3).bfloat16()
    labels = torch.randint(0, vocab, (rows,), device="cuda", generator=g)
    labels[torch.rand(rows, device="cuda", generator=g) >= live] = -100
    labels[:1] = vocab - 1
    g_rows = torch.rand(rows, device="cuda", generator=g) + 0.1
    g_rows[::9] = 0
    return x, w, labels, g_rows


def _run(x, w, labels, g_rows):
    from speculators_amd import losses as L

    xi = x.clone().requires_grad_(True)
    loss, logits = L.head_label_cross_entropy(xi, w, w.t().contiguous(), labels)
    (dx,) = torch.autograd.grad(loss, xi, g_rows)
    return loss.detach(), logits, dx


# one row, fewer rows than workgroups, a second and a third row for some; the narrowest and the widest row, a last chunk that
# is not full, one that only the first threads have
@pytest.mark.parametrize("rows,vocab", [(1, 65536), (255, 65544), (257, 151936), (600, 81920), (300, 155648)])
def test_against_two_passes_and_float64(rows, vocab, monkeypatch):
    from speculators_amd import losses as L

    x, w, labels, g_rows = _case(rows, vocab, 64, rows)
    loss, logits, dx = _run(x, w, labels, g_rows)
    monkeypatch.setattr(L, "HEAD_LOSS_ONE_PASS", False)
    loss2, logits2, dx2 = _run(x, w, labels, g_rows)
    assert torch.equal(logits, logits2)
    live = labels != -100
    assert (loss[~live] == 0).all() and (dx[~live] == 0).all() and (dx[g_rows == 0] == 0).all()
    # sums of up to 155648 fp32 exponentials in another order
    torch.testing.assert_close(loss, loss2, rtol=0, atol=4e-5)
    p = torch.softmax(logits.double(), -1)
    p[live, labels[live]] -= 1
    p[~live] = 0
    want = (p * g_rows.double().unsqueeze(1)) @ w.double()
    # the logits gradient and dx are rounded to bf16 once each: no further off than the two-pass form, which does the same
    err, err2 = (dx.double() - want).norm(), (dx2.double() - want).norm()
    assert err <= 1.1 * err2 + 1e-9 and err <= 2.0 ** -8 * want.norm() + 1e-9


def test_labels_out_of_range_and_rows_of_infinities():
    x, w, labels, g_rows = _case(40, 65536, 64, 3)
    labels[:] = torch.arange(40, device="cuda")
    labels[5], labels[6], labels[7] = 70000, -1, -100
    x[7] = float("inf")  # ignored
    x[8] = float("nan")
    g_rows[8] = 0        # weighs nothing
    loss, _, dx = _run(x, w, labels, g_rows)
    assert loss[5].isnan() and loss[6].isnan() and loss[7] == 0 and loss[8].isnan()
    keep = torch.ones(40, dtype=torch.bool, device="cuda")
    keep[[5, 6, 8]] = False
    assert torch.isfinite(loss[keep]).all() and (dx[7] == 0).all() and (dx[8] == 0).all() and torch.isfinite(dx).all()


def test_no_row_and_no_room(monkeypatch):
    from speculators_amd import losses as L

    x, w, labels, g_rows = _case(50, 65536, 64, 4)
    want = _run(x, w, labels, g_rows)
    monkeypatch.setattr(L, "LABEL_GRADIENT_SHARE", 0.0)  # no room between the forward and the backward
    got = _run(x, w, labels, g_rows)
    torch.testing.assert_close(got[0], want[0], rtol=0, atol=4e-5)
    assert (got[2].double() - want[2].double()).norm() <= 2.0 ** -7 * want[2].double().norm()
    monkeypatch.undo()
    labels[:] = -100
    loss, _, dx = _run(x, w, labels, g_rows)
    assert (loss == 0).all() and (dx == 0).all()
