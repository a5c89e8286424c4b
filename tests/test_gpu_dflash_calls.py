"""Calls of the anchored-block metrics off the common form: decay rates that are not positive."""

import pytest
import torch

from speculators_amd import losses as L
from speculators_amd import metrics as MT

pytestmark = pytest.mark.gpu

BS = 4


@pytest.mark.parametrize("gamma", [-3.0, float("inf"), 0.0, float("nan")])
@pytest.mark.parametrize("from_anchor", [False, True])
def test_decay_rates_that_are_not_positive(gamma, from_anchor):
    g = torch.Generator().manual_seed(2)
    n, vocab = 24, 96
    x, y = (torch.randn(1, n, vocab, generator=g).cuda() for _ in range(2))
    mask = (torch.rand(1, n, generator=g) < 0.8).float().cuda()
    loss, _ = MT.dflash_compute_metrics(x, y, mask, BS, gamma, sample_from_anchor=from_anchor)
    rows = L.kl_div_loss(x, y).double().reshape(-1)
    slot = torch.arange(n, device="cuda").double() % BS
    # (losses/utils.py:17-48)
    w = torch.exp(-slot / gamma) if from_anchor else torch.exp(-(slot - 1).clamp_min(0) / gamma).masked_fill(slot == 0, 0)
    want = (rows * mask.double().reshape(-1) * w).sum() / (mask.double().sum() + 1e-5)
    assert torch.isnan(want) == torch.isnan(loss)
    assert torch.isnan(want) or abs(loss.item() - want.item()) <= 2e-6 * abs(want.item())
