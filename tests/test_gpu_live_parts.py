"""Parts of a product chosen on the device for the rows that count (spx_gemm_bf16_rows_graded on the smaller tiles)."""

import pytest
import torch

pytestmark = pytest.mark.gpu


# edges of a tile row; N whole and ragged in the tiles' columns; the contraction just long enough to be cut, and ragged
@pytest.mark.parametrize("m,n,k", [(1536, 2048, 2304), (600, 1992, 2056), (96, 64, 4096)])
@pytest.mark.parametrize("live", [0, 1, 64, 65, 128, 129, 257, 1025, 5000])
def test_live_parts_against_float64(m, n, k, live):
    from speculators_amd import _lib

    lib = _lib.load()
    assert lib.spx_gemm_auto_tile(2, m, n, k, 4)
    full = lib.spx_gemm_auto_workspace_bytes(2, m, n, k, 4)
    g = torch.Generator(device="cuda").manual_seed(m + live)
    a = torch.randn(m, k, device="cuda", generator=g).bfloat16()
    b = torch.randn(n, k, device="cuda", generator=g).bfloat16()
    weight = torch.rand(m, device="cuda", generator=g) + 0.5
    rows = min(live, m)
    want = (a[:rows].double() @ b.double().t()) * weight[:rows].double().unsqueeze(1)
    # one rounding to bf16 (2^-8 of the power of two below the value) behind fp32 sums of k products
    bound = 2 ** -8 * torch.exp2(want.abs().clamp_min(1e-30).log2().floor())
    bound = bound + 2 ** -22 * (a[:rows].double().abs() @ b.double().abs().t()) * weight[:rows].double().unsqueeze(1)
    order = torch.arange(m, device="cuda", dtype=torch.int32)
    count = torch.tensor([live], dtype=torch.int32, device="cuda")
    guard = 1024
    got = []
    for nbytes in (full, full):
        ws = torch.full((nbytes // 4 + guard,), 3.0, device="cuda")
        c = torch.full((m, n), 2.0, dtype=torch.bfloat16, device="cuda")
        _lib.call("spx_gemm_bf16_rows_graded", a, k, b, k, c, n, m, n, k, count, order, weight, torch.ones((), device="cuda"), 1.0,
                  4, 4, ws, nbytes, _lib.stream_ptr(a.device))
        assert (ws[nbytes // 4:] == 3).all() and (c[rows:] == 2).all()
        assert rows == 0 or ((c[:rows].double() - want).abs() <= bound).all()
        got.append(c)
    assert torch.equal(*got)
