"""Grouped products whose rows are picked out of a larger matrix, against the same products on a copy of those rows."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _case(sizes, tokens, seed):
    g = torch.Generator().manual_seed(seed)
    rows = sum(sizes)
    src = torch.randint(0, tokens, (rows,), generator=g, dtype=torch.int32)
    src[::7] = -1  # numbers outside of the matrix: rows of zeros
    src[3::11] = tokens
    off = torch.tensor([0] + sizes).cumsum(0).to(torch.int32)
    return g, rows, src, off


def _copy(x, src):
    inside = (src >= 0) & (src < x.shape[0])
    return torch.where(inside[:, None], x[src.clamp(0, x.shape[0] - 1).long()], torch.zeros((), dtype=x.dtype))


# edges of an 8-row load group, a K step, a slab and a tile; contractions with one and with three slab buffers
@pytest.mark.parametrize("sizes,n,k", [([1, 7, 8, 9, 0, 127, 128, 129], 264, 72), ([5] * 600, 520, 1024), ([3] * 30, 264, 1032)])
@pytest.mark.parametrize("form", [0, 1])
def test_rows_of_the_first_operand(sizes, n, k, form):
    from speculators_amd import moe

    g, rows, src, off = _case(sizes, 61, n + k)
    x = torch.randn(61, k, generator=g).bfloat16()
    w = torch.randn(len(sizes), *((n, k) if form == 0 else (k, n)), generator=g).bfloat16().cuda()
    p = moe._Picked(src.cuda(), off.cuda())
    got = p.rows_of(form, x.cuda(), w, True)
    plain = moe.gemm_nt_grouped if form == 0 else moe.gemm_nn_grouped
    want = plain(_copy(x, src).cuda(), w, off.cuda())
    assert torch.equal(got, want)  # the same tiles, in the same order
    # the table is there already; rows as they lie
    assert torch.equal(p.rows_of(form, _copy(x, src).cuda(), w, False), want)


@pytest.mark.parametrize("sizes,m,n", [([1, 31, 32, 33, 0, 63, 64, 65, 127, 129, 300], 136, 264), ([200], 128, 8)])
@pytest.mark.parametrize("operand", [0, 1])
@pytest.mark.parametrize("fp32", [False, True])
@pytest.mark.parametrize("accumulate", [False, True])
def test_rows_of_a_weight_gradient(sizes, m, n, operand, fp32, accumulate):
    from speculators_amd import moe

    g, rows, src, off = _case(sizes, 45, m + n)
    tokens = torch.randn(45, (m, n)[operand], generator=g).bfloat16()
    other = torch.randn(rows, (n, m)[operand], generator=g).bfloat16().cuda()
    fill = torch.randn(len(sizes) + 1, m, n, generator=g).to(torch.float32 if fp32 else torch.bfloat16).cuda()
    out, want = fill.clone(), fill.clone()
    pair = (tokens.cuda(), other) if operand == 0 else (other, tokens.cuda())
    moe._Picked(src.cuda(), off.cuda()).weight_gradient(*pair, operand, out[:-1], accumulate)
    copy = _copy(tokens, src).cuda()
    moe.gemm_tn_grouped(*((copy, other) if operand == 0 else (other, copy)), off.cuda(), want[:-1], accumulate=accumulate)
    assert torch.equal(out, want)
    assert torch.equal(out[-1], fill[-1])


def test_refused():
    from speculators_amd import _lib, moe

    x, w = torch.zeros(4, 16, device="cuda", dtype=torch.bfloat16), torch.zeros(1, 8, 16, device="cuda", dtype=torch.bfloat16)
    p = moe._Picked(torch.zeros(300, device="cuda", dtype=torch.int32), torch.tensor([0, 300], device="cuda", dtype=torch.int32))
    with pytest.raises(_lib.SpxError, match="256 rows a group"):
        p.rows_of(0, x, w, True)
    with pytest.raises(ValueError, match="shape mismatch"):
        p.rows_of(1, x, w, True)
