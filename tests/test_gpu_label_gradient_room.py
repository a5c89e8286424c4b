"""Logits gradients that wait for the backward: as many steps of a forward as the memory that is left allows, no more."""

import pytest
import torch

pytestmark = pytest.mark.gpu

TOKENS, VOCAB, STEPS = 2003, 65536, 3
ROWS = TOKENS - STEPS - 1
LOGITS = ROWS * VOCAB * 2  # bytes of one step


def _model():
    from speculators_amd.mtp import MTPConfig, MTPDraftModel

    torch.manual_seed(0)
    model = MTPDraftModel(MTPConfig(hidden_size=128, num_attention_heads=2, num_key_value_heads=1, head_dim=64,
                                    intermediate_size=256, vocab_size=VOCAB, num_speculative_steps=STEPS)).bfloat16().cuda()
    ids = torch.randint(0, VOCAB, (1, TOKENS), device="cuda")
    hs = torch.randn(1, TOKENS, 128, device="cuda").bfloat16()
    model(ids, hs)[1].backward()  # (kept copies of frozen weights and workspaces are there from here on)
    model.zero_grad(set_to_none=True)
    return model, ids, hs


def _pass(model, ids, hs, monkeypatch, memory=None):
    """``(loss, gradients, one-read passes, peak bytes over what was there)`` with ``memory`` bytes to allocate."""
    from speculators_amd import _lib
    from speculators_amd import losses as L

    taken, call = [], _lib.call
    monkeypatch.setattr(_lib, "call", lambda name, *a: (taken.append(name), call(name, *a))[1])
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    if memory is not None:
        monkeypatch.setattr(L, "_available_memory", lambda device: before + memory - torch.cuda.memory_allocated())
    _, loss, _ = model(ids, hs)
    loss.backward()
    monkeypatch.undo()
    grads = [p.grad for p in model.parameters() if p.grad is not None]
    model.zero_grad(set_to_none=True)
    return loss.detach(), grads, taken.count("spx_label_ce_fwd_grad"), torch.cuda.max_memory_allocated() - before


# bytes in logits of one step: nothing is kept; the first step's two successors are (what is there is 10, then 9 less the
# layer's activations, then 7); all three are
@pytest.mark.parametrize("memory,kept", [(5.5, 0), (10.5, 2), (40, 3)])
def test_steps_within_the_memory_that_is_left(memory, kept, monkeypatch):
    from speculators_amd import losses as L

    model, ids, hs = _model()
    loss, grads, passes, peak = _pass(model, ids, hs, monkeypatch, int(memory * LOGITS))
    assert passes == kept and peak <= memory * LOGITS
    monkeypatch.setattr(L, "HEAD_LOSS_ONE_PASS", False)
    want_loss, want, none, _ = _pass(model, ids, hs, monkeypatch)
    assert none == 0 and len(grads) == len(want) and len(want) > 8
    torch.testing.assert_close(loss, want_loss, rtol=1e-5, atol=0)  # (fp32 sums in another order)
    for a, b in zip(grads, want, strict=True):
        # the row weight in front of or behind the gradient's rounding to bf16 (2^-8 in dx), and the roundings of a dozen
        # tensors between it and a weight's gradient that fall the other way: sqrt(12) 2^-8
        assert (a.double() - b.double()).norm() <= 2.0 ** -6 * b.double().norm()


def test_memory_that_is_left(monkeypatch):
    """What the process can still allocate: with the card's, and with a share of it."""
    from speculators_amd import losses as L

    device = torch.device("cuda", torch.cuda.current_device())
    block = torch.empty(1 << 28, device=device, dtype=torch.uint8)
    total = torch.cuda.mem_get_info()[1]
    left = L._available_memory(device)
    assert 0 < left <= total - torch.cuda.memory_allocated()
    del block  # (held by the allocator now: can be allocated again)
    assert abs(L._available_memory(device) - left - (1 << 28)) < 1 << 27
    try:
        torch.cuda.set_per_process_memory_fraction(0.5)
        assert L._available_memory(device) <= total // 2 - torch.cuda.memory_allocated()
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)


def test_room_is_shared_by_the_calls_of_a_forward(monkeypatch):
    from speculators_amd import losses as L

    rows = torch.empty(4, 1024, device="cuda", dtype=torch.bfloat16)  # 8 KB
    monkeypatch.setattr(L, "_available_memory", lambda device: 4 * 2 * 8192)
    assert L.GradientRoom().take(rows) is not None
    room = L.GradientRoom(3)
    assert [room.take(rows) is not None for _ in range(4)] == [False, True, True, True]
    monkeypatch.setattr(L, "_available_memory", lambda device: 4 * 8192 - 1)
    assert L.GradientRoom().take(rows) is None
