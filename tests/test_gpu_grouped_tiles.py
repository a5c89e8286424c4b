"""The tiles the grouped products choose between (csrc/gemm_tile.hip), at the sizes where each can go wrong: groups at the
edges of a K step (32), a slab (64) and a tile, ragged result edges, both sides of every rule."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _offsets(sizes):
    return torch.tensor([0] + sizes).cumsum(0).to(torch.int32)


# (up to 512 rows a group on average: 128 x 128 tiles with one slab; above: 256 x 256)
@pytest.mark.parametrize("sizes,m,n", [([1, 31, 32, 33, 0, 63, 64, 65, 95, 96, 97, 127, 129, 600], 136, 264),
                                       ([512], 128, 128), ([513], 264, 8), ([1000, 30, 1100], 136, 392)])
@pytest.mark.parametrize("fp32", [False, True])
def test_weight_gradient_tiles(sizes, m, n, fp32):
    from speculators_amd.moe import gemm_tn_grouped

    g = torch.Generator().manual_seed(len(sizes) + m)
    a, b = (torch.randn(sum(sizes) + 5, c, generator=g).bfloat16() for c in (m, n))
    a[sum(sizes):] = float("nan")  # rows of no group are not read into anything
    out = torch.full((len(sizes) + 1, m, n), 3.0, dtype=torch.float32 if fp32 else torch.bfloat16, device="cuda")
    gemm_tn_grouped(a.cuda(), b.cuda(), _offsets(sizes).cuda(), out[:-1])
    assert (out[-1] == 3).all()
    # fp32 sums of products of rounded operands in another order / one rounding to bf16
    tol = 2e-6 * max(sizes) ** 0.5 if fp32 else 2 ** -8
    at = 0
    for e, rows in enumerate(sizes):
        want = a[at:at + rows].double().t() @ b[at:at + rows].double()
        err = (out[e].double().cpu() - want).abs().max().item()
        assert err <= tol * max(want.abs().max().item(), 1.0), (e, rows, err)
        at += rows


# (contractions up to 1024 with four tiles for every compute unit: one slab, two workgroups a compute unit)
@pytest.mark.parametrize("groups,n,k", [(1024, 40, 8), (1024, 40, 72), (520, 264, 1024), (520, 264, 1032), (511, 264, 96)])
@pytest.mark.parametrize("transposed", [False, True])
def test_expert_product_tiles(groups, n, k, transposed):
    from speculators_amd.moe import gemm_nn_grouped, gemm_nt_grouped

    g = torch.Generator().manual_seed(groups + k)
    sizes = torch.randint(0, 12, (groups,), generator=g)
    sizes[5], sizes[6], sizes[7] = 128, 129, 257
    sizes = sizes.tolist()
    a = torch.randn(sum(sizes), k, generator=g).bfloat16().cuda()
    w = torch.randn(groups, n, k, generator=g).bfloat16().cuda()
    out = torch.full((sum(sizes) + 3, n), 7.0, dtype=torch.bfloat16, device="cuda")
    if transposed:
        gemm_nn_grouped(a, w.transpose(1, 2).contiguous(), _offsets(sizes).cuda(), out=out[:-3])
    else:
        gemm_nt_grouped(a, w, _offsets(sizes).cuda(), out=out[:-3])
    assert (out[-3:] == 7).all()
    at = 0
    for e, rows in enumerate(sizes):
        if rows:
            want = a[at:at + rows].float() @ w[e].float().t()
            assert (out[at:at + rows].float() - want).abs().max() <= 2 ** -8 * want.abs().max() + 1e-3, (e, rows)
        at += rows


@pytest.mark.parametrize("sizes,n,k", [([300, 700, 0, 256], 264, 520), ([257], 8, 1024)])
def test_tall_tiles_of_the_forward_product(sizes, n, k):
    """More than 256 rows a group on average."""
    from speculators_amd.moe import gemm_nt_grouped

    g = torch.Generator().manual_seed(n)
    a = torch.randn(sum(sizes), k, generator=g).bfloat16().cuda()
    w = torch.randn(len(sizes), n, k, generator=g).bfloat16().cuda()
    got = gemm_nt_grouped(a, w, _offsets(sizes).cuda())
    at = 0
    for e, rows in enumerate(sizes):
        if rows:
            want = a[at:at + rows].float() @ w[e].float().t()
            assert (got[at:at + rows].float() - want).abs().max() <= 2 ** -8 * want.abs().max() + 1e-3, (e, rows)
        at += rows
