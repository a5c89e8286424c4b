"""The tiles of 192 rows of spx_gemm_bf16_auto (192 x 256 in both forms, 192 x 192 and 192 x 128 in one): ragged rows, columns and
contractions, parts, padded and unaligned results, and a device count of rows."""

import pytest
import torch

pytestmark = pytest.mark.gpu

SHAPES = [  # (form, tile, M, N, K)
    (0, 4, 2903, 3080, 1032), (0, 4, 2305, 4083, 1032), (0, 5, 2689, 3080, 520), (0, 5, 1537, 5117, 1032), (0, 5, 1300, 3080, 4104),
    (1, 4, 2903, 4088, 1032), (1, 4, 1537, 6152, 1032), (1, 6, 1300, 3080, 1032), (1, 6, 2689, 1544, 1032), (1, 6, 190, 10248, 4104)]


def test_forward_projections_on_192_x_192_tiles():
    from speculators_amd import gemm

    # (rows, N, K): two rounds, one round, more than two rounds (library), 192 x 256 tiles (library)
    for m, n, k, own in ((3001, 6144, 8192, True), (2900, 3072, 4096, True), (1300, 57344, 8192, False), (3001, 4096, 4096, False)):
        assert gemm._own_forward(m, n, k) == own, (m, n, k)


@pytest.mark.parametrize("form,tile,m,n,k", SHAPES)
@pytest.mark.parametrize("pad", [0, 8, 3])
@pytest.mark.parametrize("live", [None, 0, 1, 193, 5000])
def test_product_against_float64(form, tile, m, n, k, pad, live):
    from speculators_amd import _lib

    lib = _lib.load()
    plan = 2 if form == 0 and live is not None else form  # (with a count of rows that form stays with the other tiles)
    assert plan == 2 or lib.spx_gemm_auto_tile(form, m, n, k, 4) == tile
    assert lib.spx_gemm_auto_tile(2, m, n, k, 4) < 4
    g = torch.Generator(device="cuda").manual_seed(m + n)
    a = torch.randn(m, k + 8, device="cuda", generator=g).bfloat16()[:, :k]
    b = torch.randn(*((n, k + 8) if form == 0 else (k, n + 8)), device="cuda", generator=g).bfloat16()
    b = b[:, :k] if form == 0 else b[:, :n]
    rows = m if live is None else min(live, m)
    x = a[:rows].double()
    want = x @ (b.double().t() if form == 0 else b.double())
    nbytes = lib.spx_gemm_auto_workspace_bytes(plan, m, n, k, 4)
    ws = torch.empty(nbytes // 4, device="cuda", dtype=torch.float32) if nbytes else None
    m_live = None if live is None else torch.tensor([live], dtype=torch.int32, device="cuda")
    got = []
    for _ in range(2):
        c = torch.full((m, n + pad), 2.0, dtype=torch.bfloat16, device="cuda")
        _lib.call("spx_gemm_bf16_auto", form, a, a.stride(0), b, b.stride(0), c, c.stride(0), m, n, k, m_live, 4, ws, nbytes,
                  _lib.stream_ptr(a.device))
        got.append(c)
    assert torch.equal(got[0], got[1])
    # (fp32 sums of k products, one rounding to bf16)
    assert rows == 0 or (got[0][:rows, :n].double() - want).abs().max().item() <= 2 ** -8 * want.abs().max().item() + 1e-4
    assert (got[0][:, n:] == 2).all() and (got[0][rows:] == 2).all()
