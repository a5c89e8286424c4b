"""Tokens that the experts take: column slices of a wide buffer, and tokens that the caller writes to afterwards."""

import pytest
import torch

pytestmark = pytest.mark.gpu

E, H, I, K = 4, 64, 32, 2


def _parts(tokens, seed=0):
    g = torch.Generator().manual_seed(seed)
    gate_up = torch.nn.Parameter((torch.randn(E, 2 * I, H, generator=g) / 8).bfloat16().cuda())
    down = torch.nn.Parameter((torch.randn(E, H, I, generator=g) / 8).bfloat16().cuda())
    x = torch.randn(tokens, H, generator=g).bfloat16().cuda()
    idx = torch.stack([torch.randperm(E, generator=g)[:K] for _ in range(tokens)]).cuda()
    scores = torch.rand(tokens, K, generator=g).cuda()
    return gate_up, down, x, scores, idx


def _staged(gate_up, down):
    from speculators_amd.weights import WeightStager

    stager = WeightStager()
    stager.begin(uses=1)
    return stager.get(gate_up), stager.get(down)


# (16777216: 70 rows of the slice span more than 32-bit offsets reach)
@pytest.mark.parametrize("width", [H + 8, 1 << 24])
@pytest.mark.parametrize("grad", [False, True])
def test_column_slice(width, grad):
    from speculators_amd import moe

    gate_up, down, x, scores, idx = _parts(70)
    wide = torch.empty(70, width, device="cuda", dtype=torch.bfloat16)
    wide[:, :H] = x
    got = []
    with torch.set_grad_enabled(grad):
        for x2 in (x, wide[:, :H]):
            y = moe.experts_mlp(x2, scores, idx, *_staged(gate_up, down))
            got.append([y, *(torch.autograd.grad(y, (gate_up, down), torch.ones_like(y)) if grad else ())])
    assert all(torch.equal(a, b) for a, b in zip(*got, strict=True))


@pytest.mark.parametrize("trains", [True, False])
def test_tokens_written_to_before_the_backward(trains):
    from speculators_amd import moe

    gate_up, down, x, scores, idx = _parts(70)
    gate_up.requires_grad_(trains)
    x.requires_grad_(True)
    leaves = (x, gate_up, down) if trains else (x, down)
    got = []
    for write in (False, True):
        x2 = x * 1.0
        y = moe.experts_mlp(x2, scores, idx, *_staged(gate_up, down))
        if write:
            x2.zero_()
        got.append(torch.autograd.grad(y, leaves, torch.ones_like(y)))
    assert all(torch.equal(a, b) for a, b in zip(*got, strict=True))
