"""Logits of several steps that the node of all TTT steps holds at a time: within their bound, fewer where memory is short."""

import pytest
import torch

pytestmark = pytest.mark.gpu

T, VOCAB, H, STEPS = 1024, 32768, 64, 4
LOGITS = T * VOCAB * 2  # bytes of one step


def _run(x, w, y, mask, grad, memory=None):
    """``(loss, tokens, gradients, peak bytes of the forward over what was there)`` with ``memory`` bytes to allocate."""
    from speculators_amd import metrics as MT

    xs = [v.clone().requires_grad_(grad) for v in x]
    wt = w.t().contiguous()
    run = MT.TTTSteps.take(xs[0], w, y, mask, mask.clone(), STEPS, 0.8, None)
    for v in xs:
        run.add(v)
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    torch.cuda.reset_peak_memory_stats()
    before, total = torch.cuda.memory_allocated(), torch.cuda.mem_get_info()[1]
    try:
        if memory is not None:
            torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + memory) / total)
        loss, _, tokens = run.finish(w, wt)
        peak = torch.cuda.max_memory_allocated() - before
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
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
    # all four do not fit, nor do three
    short = _run(*case, memory=gradient + 2.5 * LOGITS)
    monkeypatch.setattr(L, "STEPS_LOGITS_BYTES", LOGITS)
    one = _run(*case)
    assert one[3] < gradient + 1.5 * LOGITS
    for got in (short, one):  # a row's arithmetic does not depend on the rows beside it
        assert torch.equal(got[0], want[0]) and all(torch.equal(a, b) for a, b in zip(got[1], want[1], strict=True))
        assert all(torch.equal(a, b) for a, b in zip(got[2], want[2], strict=True))
    monkeypatch.undo()
    with pytest.raises(torch.OutOfMemoryError):
        _run(*case, memory=gradient + 0.5 * LOGITS)
