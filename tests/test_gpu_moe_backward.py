"""The backward of the experts' SwiGLU with the router's weight in it (``spx_moe_swiglu_bwd``) against float64."""

import pytest
import torch

pytestmark = pytest.mark.gpu


# one chunk of a row; a whole trip of a wave (512 columns), one chunk more, two trips; rows that do not fill a workgroup
@pytest.mark.parametrize("rows,inter", [(1, 8), (3, 512), (6, 520), (130, 1024)])
@pytest.mark.parametrize("score_dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("full", [True, False])
def test_weighted_swiglu_backward(rows, inter, score_dtype, full):
    from speculators_amd import _lib

    g = torch.Generator().manual_seed(rows + inter)
    hid = torch.randn(rows, 2 * inter, generator=g).bfloat16()
    d = torch.randn(rows, inter, generator=g).bfloat16()
    s = torch.rand(rows, generator=g)
    order = torch.randperm(rows, generator=g)
    dh = torch.full((rows, 2 * inter), 9.0, dtype=torch.bfloat16, device="cuda")
    act = torch.full((rows, inter), 9.0, dtype=torch.bfloat16, device="cuda") if full else None
    ds = torch.full((rows,), 9.0, dtype=score_dtype, device="cuda") if full else None
    _lib.call("spx_moe_swiglu_bwd", hid.cuda(), 2 * inter, order.cuda(), s.cuda(), d.cuda(), inter, dh, 2 * inter, act, inter,
              ds, int(score_dtype == torch.float32), rows, inter, _lib.stream_ptr(dh.device))
    x = hid.double().requires_grad_(True)
    gate, up = x.chunk(2, dim=-1)
    plain = torch.nn.functional.silu(gate) * up
    w = s.double()[order, None]
    (want,) = torch.autograd.grad((plain * w * d.double()).sum(), x)
    # one rounding to bf16 of fp32 products (dh); of the rounded silu's product (act): two
    assert (dh.double().cpu() - want).abs().max() <= 2 ** -8 * want.abs().max()
    if full:
        assert (act.double().cpu() - plain * w).abs().max() <= 2 ** -7 * (plain * w).abs().max()
        ref = (plain * d.double()).sum(-1)
        # a silu rounding (2^-9 of each term) and the result's own
        bound = 2 ** -9 * (plain * d.double()).abs().sum(-1) + 2 ** -8 * ref.abs() + 1e-5
        got = ds.double().cpu()[order]
        assert ((got - ref).abs() <= bound).all()
