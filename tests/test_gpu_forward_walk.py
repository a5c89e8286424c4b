"""Forward projections that workgroups walk: rows and weights as callers hand them over, aligned or not."""

import pytest
import torch

pytestmark = pytest.mark.gpu


class _Weight:
    trainable = False

    def __init__(self, w):
        self.w = w


# a short contraction, a cut last round; (rows' padding, their offset, the weight's offset in elements)
@pytest.mark.parametrize("m,n,k", [(2900, 8200, 512), (2900, 16640, 4096)])
@pytest.mark.parametrize("pad,off,w_off", [(0, 0, 0), (8, 8, 8), (3, 0, 0), (8, 1, 0), (0, 0, 3)])
def test_projection(m, n, k, pad, off, w_off):
    from speculators_amd import gemm

    assert gemm._walking_forward(m, n, k) and not gemm._own_forward(m, n, k)
    g = torch.Generator(device="cuda").manual_seed(m + pad)
    x = torch.randn(m * (k + pad) + off, device="cuda", generator=g).bfloat16()[off:].view(m, k + pad)[:, :k]
    w = torch.randn(n * k + w_off, device="cuda", generator=g).bfloat16()[w_off:].view(n, k)
    aligned = pad % 8 == 0 and off % 8 == 0 and w_off % 8 == 0
    assert (gemm._rows_in_lines(x) and gemm._rows_in_lines(w)) == aligned
    got = gemm.linear_staged(x.unsqueeze(0), _Weight(w))[0].double()
    want = x.double() @ w.double().T
    # one rounding to bf16 and fp32 sums of k terms of order one
    assert ((got - want).abs() <= 2.0 ** -8 * want.abs() + k * 2.0 ** -24 * 8 * k ** 0.5).all()
