"""The node that stages a layer's weights together (weights._StageAll), without a GPU: which weights' gradients a backward pass forms."""

import pytest
import torch

from speculators_amd import _lib, weights


class _Records:
    """Stands for ``weights._Uses``: one use a pass, whose weight gradient is ``value`` everywhere."""

    def __init__(self, shape, value, formed):
        self.shape, self.value, self.formed = shape, value, formed

    def sole(self):
        return None

    def finish(self, bf16_ok=False):
        self.formed.append(self.value)
        return torch.full(self.shape, float(self.value))

    def drop(self):
        pass


class _Use(torch.autograd.Function):
    """A product against every staged weight, as a layer's node: it reaches all of their tokens."""

    @staticmethod
    def forward(ctx, x, *tokens):
        ctx.shapes = [t.shape for t in tokens]
        return x * 2

    @staticmethod
    def backward(ctx, g):
        return (g * 2, *(torch.zeros(()).expand(s) for s in ctx.shapes))


def _layer():
    groups = [tuple(torch.nn.Parameter(torch.ones(r, 8)) for r in rows) for rows in ((2, 1), (3,), (4, 4))]
    groups[0][1].requires_grad_(False)
    formed = []
    records = [_Records((sum(p.shape[0] for p in g), 8), i + 1, formed) for i, g in enumerate(groups)]
    out = weights._StageAll.apply(records, {}, [len(g) for g in groups], *(p for g in groups for p in g))
    x = torch.ones(4, requires_grad=True)
    return groups, formed, x, _Use.apply(x, *out[1::2]).sum()


def test_every_weight_of_a_whole_backward():
    groups, formed, x, loss = _layer()
    loss.backward()
    assert formed == [1, 2, 3] and x.grad is not None
    for i, g in enumerate(groups):
        for p in g:
            assert (p.grad is None) if not p.requires_grad else (p.grad == i + 1).all()


@pytest.mark.parametrize("asked,form", [((0, 0), [1]), ((1, 0), [2]), ((2, 1), [3]), (None, [])])
@pytest.mark.parametrize("grad", [True, False])
def test_only_the_weights_that_are_asked_for(asked, form, grad):
    groups, formed, x, loss = _layer()
    wanted = x if asked is None else groups[asked[0]][asked[1]]
    if grad:
        got, = torch.autograd.grad(loss, (wanted,), retain_graph=True)
    else:
        loss.backward(inputs=(wanted,), retain_graph=True)
        got = wanted.grad
    assert formed == form and (got == (2 if asked is None else form[0])).all()
    assert sum(p.grad is not None for g in groups for p in g) == (0 if grad or asked is None else 1)
    # the rest is there for the next pass
    loss.backward()
    assert formed == form + [1, 2, 3]


def test_a_weight_behind_other_nodes():
    """Parameters that are no leaves: asked for by themselves and by what they are made from."""
    made = [torch.nn.Parameter(torch.ones(2, 8)) for _ in range(2)]
    inner = [p * 3 for p in made]
    formed = []
    out = weights._StageAll.apply([_Records((2, 8), i + 1, formed) for i in range(2)], {}, [1, 1], *inner)
    loss = _Use.apply(torch.ones(4), *out[1::2]).sum()
    got, = torch.autograd.grad(loss, (made[1],), retain_graph=True)
    assert formed == [2] and (got == 6).all()
    got, = torch.autograd.grad(loss, (inner[0],))
    assert formed == [2, 1] and (got == 1).all()


def test_wanted_takes_contexts_alone():
    for wrong in (torch.ones(2), None, object()):
        with pytest.raises(TypeError, match="context"):
            _lib.native().wanted(wrong)


class _Product(torch.autograd.Function):
    """``x @ w.T`` that leaves its weight gradient to the staging node, as ``gemm._StagedLinear``."""

    @staticmethod
    def forward(ctx, x, w, _token, records):
        ctx.save_for_backward(x, w)
        ctx.records = records
        return x @ w.T

    @staticmethod
    def backward(ctx, dy):
        x, w = ctx.saved_tensors
        return dy @ w, None, ctx.records.defer(-1, dy, x), None


def _two_products(monkeypatch):
    monkeypatch.setattr(weights, "wgrad_product", lambda dy, x, acc: dy.T @ x if acc is None else acc + dy.T @ x)
    a, b = (torch.nn.Parameter(torch.randn(6, 8)) for _ in range(2))
    records = [weights._Uses(1, False) for _ in range(2)]
    out = weights._StageAll.apply(records, {i: w.detach() for i, w in enumerate((a, b))}, [1, 1], a, b)
    for r, token in zip(records, out[1::2], strict=True):
        r.shape, r.device, r.trainable = token.shape, token.device, True
    x = torch.randn(5, 8, requires_grad=True)
    return a, b, x, [_Product.apply(x, out[2 * i], out[2 * i + 1], records[i]).square().sum() for i in range(2)]


def test_records_of_an_earlier_pass_are_not_used(monkeypatch):
    """A pass for the input alone leaves what the uses recorded; the next one, which reaches the node by one of the two, forms that
    one's gradient and no other."""
    a, b, x, (loss_a, loss_b) = _two_products(monkeypatch)
    torch.autograd.grad(loss_a + loss_b, (x,), retain_graph=True)
    loss_a.backward(retain_graph=True)
    assert b.grad is None
    torch.testing.assert_close(a.grad, 2 * (x @ a.T).T @ x)
    a.grad = None
    (loss_a + loss_b).backward()
    for p in (a, b):
        torch.testing.assert_close(p.grad, 2 * (x @ p.T).T @ x)
