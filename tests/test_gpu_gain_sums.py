"""Gradients of RMSNorm gains: many partial-sum buffers reduced in one launch (``spx_rmsnorm_dweights``, sixteen to a launch), and
gains staged together (``WeightStager.gains``) against each staged alone."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("count", [1, 2, 16, 17, 33])
def test_sums_of_many_gains(count):
    from speculators_amd import _lib

    g = torch.Generator().manual_seed(count)
    widths, heights = [8, 40, 64, 128, 2048, 4096, 16384], [1, 5, 127, 128, 129, 512, 1024]
    parts, args = [], []
    for i in range(count):
        h, slots = widths[(3 * i + count) % 7], heights[(2 * i + count) % 7]
        parts.append(torch.randn(slots, h, generator=g))
        args += [parts[-1].cuda(), slots, h, i % 2]
    out = _lib.native().gain_sums(*args)
    assert len(out) == count
    for i, (part, got) in enumerate(zip(parts, out)):
        want, size = part.double().sum(0), part.double().abs().sum(0)
        assert got.dtype == (torch.float32 if i % 2 else torch.bfloat16) and got.shape == want.shape
        # fp32 sums of `slots` values in chains of at most slots / 128 + 24; a rounding to bf16 on top
        bound = (part.shape[0] / 128 + 25) * 2.0 ** -24 * size + (0 if i % 2 else 2.0 ** -8) * want.abs()
        assert ((got.double().cpu() - want).abs() <= bound).all(), i


@pytest.mark.parametrize("master", [False, True])
def test_gains_staged_together_equal_gains_staged_alone(master):
    """Bit for bit, with a gain that is used twice, one that is not used, one that also gets a gradient the ordinary way, a
    frozen one, and a second backward over the same graph."""
    from speculators_amd import fused_ops as FO
    from speculators_amd.weights import WeightStager

    h, rows = 256, 300
    g = torch.Generator().manual_seed(9)
    values = [1 + 0.2 * torch.randn(h, generator=g) for _ in range(6)]
    x = torch.randn(1, rows, h, generator=g).bfloat16().cuda()
    weights = [torch.randn(1, rows, h, generator=g).cuda() for _ in range(4)]

    class Norm:
        def __init__(self, v, trains=True):
            self.weight = v.cuda().to(torch.float32 if master else torch.bfloat16).requires_grad_(trains)

    def run(together):
        norms = [Norm(v, trains=i != 5) for i, v in enumerate(values)]
        stager = WeightStager()
        stager.begin()
        with torch.autocast("cuda", dtype=torch.bfloat16, enabled=master):
            if together:
                stager.gains(norms)
            w = [stager.gain(n.weight) for n in norms]
            assert not w[5].requires_grad
            y = FO.rms_norm(FO.rms_norm(x, w[0], 1e-5), w[1], 1e-5)
            z = FO.rms_norm(y, w[0], 1e-5)
            outs = [y, z, FO.rms_norm(z, w[2], 1e-5) + w[2], FO.rms_norm(z, w[5], 1e-5)]
        total = sum((o.float() * k).sum() for o, k in zip(outs, weights))
        total.backward(retain_graph=True)
        first = [n.weight.grad.clone() if n.weight.grad is not None else None for n in norms]
        for n in norms:
            n.weight.grad = None
        (only,) = torch.autograd.grad(total, norms[1].weight, retain_graph=True)
        assert torch.equal(only, first[1]) and norms[0].weight.grad is None
        total.backward()
        assert all((n.weight.grad is None) == (f is None) and (f is None or torch.equal(n.weight.grad, f))
                   for n, f in zip(norms, first))
        return first

    one, all_ = run(False), run(True)
    assert one[3] is None and one[4] is None and one[5] is None and one[2] is not None
    for a, b in zip(one, all_):
        assert (a is None) == (b is None) and (a is None or (a.dtype == b.dtype and torch.equal(a, b)))
