"""Logits of several steps that the node of all TTT steps holds at a time: within their bound, fewer where memory is short."""

import weakref

import pytest
import torch

pytestmark = pytest.mark.gpu

T, VOCAB, H, STEPS = 1024, 32768, 64, 4
LOGITS = T * VOCAB * 2  # bytes of one step


def _run(x, w, y, mask, grad, held=STEPS):
    """``(loss, tokens, gradients, peak bytes of the forward over what was there)``; an allocation fails where logits of
    ``held`` steps are there already."""
    from speculators_amd import gemm
    from speculators_amd import metrics as MT

    xs = [v.clone().requires_grad_(grad) for v in x]
    wt = w.t().contiguous()
    run = MT.TTTSteps.take(xs[0], w, y, mask, mask.clone(), STEPS, 0.8, None)
    for v in xs:
        run.add(v)
    product, made = gemm.matmul_nt, []

    def matmul_nt(*a, **kw):
        if sum(m() is not None for m in made) >= held:
            raise torch.OutOfMemoryError("no room for the logits of one more step")
        out = product(*a, **kw)
        made.append(weakref.ref(out))
        return out

    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    with pytest.MonkeyPatch.context() as m:
        m.setattr(gemm, "matmul_nt", matmul_nt)
        loss, _, tokens = run.finish(w, wt)
    peak = torch.cuda.max_memory_allocated() - before
    return loss.detach(), tokens, torch.autograd.grad(loss, xs) if grad else (), peak


@pytest.mark.parametrize("grad", [False, True])
def test_logits_of_a_few_steps_at_a_time(grad, monkeypatch):
    from speculators_amd import losses as L

    g = torch.Generator(device="cuda").manual_seed(0)
    x = [torch.randn(1, T, H, device="cuda", generator=g).bfloat16() for _ in range(STEPS)]
    w = (torch.randn(VOCAB, H, device="cuda", generator=g) * 0.4).bfloat16()
    y = torch.randn(1, T, VOCAB, device="cuda", generator=g).bfloat16()
    mask = (torch.rand(1, T, device="cuda", generator=g) < 0.7).float()
    case = (x, w, y, mask, grad)
    gradient = STEPS * LOGITS if grad else 0
    _run(*case)
    want = _run(*case)
    assert want[3] >= gradient + STEPS * LOGITS
    got = [_run(*case, held=n) for n in (3, 1)]  # two steps at a time, one
    monkeypatch.setattr(L, "STEPS_LOGITS_BYTES", LOGITS)
    got.append(_run(*case))
    assert got[1][3] < gradient + 1.5 * LOGITS and got[2][3] < gradient + 1.5 * LOGITS
    for loss, tokens, grads, _ in got:  # a row's arithmetic does not depend on the rows beside it
        assert torch.equal(loss, want[0]) and all(torch.equal(a, b) for a, b in zip(tokens, want[1], strict=True))
        assert all(torch.equal(a, b) for a, b in zip(grads, want[2], strict=True))
    with pytest.raises(torch.OutOfMemoryError):
        _run(*case, held=0)
