"""Norms that add the parts of a cut product themselves, against the product's own last pass and the norm behind it."""

import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


# every form of the norm kernels (a wave a row, 256, 512 and 1024 threads), one row, ragged rows, one to eight parts; rows
# on both sides of the 1024 row slots of the backward
@pytest.mark.parametrize("rows,h", [(1, 8), (7, 512), (333, 520), (512, 2048), (1500, 2056), (65, 4096), (9, 8192), (5, 16384)])
@pytest.mark.parametrize("parts", [1, 2, 3, 8])
def test_sum_of_parts_in_the_norm(rows, h, parts):
    from speculators_amd import _lib

    g = torch.Generator(device="cuda").manual_seed(rows + parts)
    r = lambda *s: torch.randn(*s, device="cuda", generator=g)  # noqa: E731
    partial, a, gain, dres = r(parts, rows, h), r(rows, h).bfloat16(), r(h).bfloat16(), r(rows, h).bfloat16()
    st = _lib.stream_ptr(a.device)
    total = torch.zeros(rows, h, device="cuda")
    for p in partial:  # (the order of the kernel)
        total += p
    b = total.bfloat16()
    # forward: bit for bit the norm of the rounded sum
    got, want = [[torch.empty_like(a), torch.empty_like(a), torch.empty(rows, device="cuda")] for _ in range(2)]
    _lib.call("spx_add_rmsnorm_fwd", a, h, b, h, want[0], h, gain, want[1], h, want[2], rows, h, 1e-6, st)
    _lib.call("spx_add_rmsnorm_fwd_parts", a, h, partial, parts, got[0], h, gain, got[1], h, got[2], rows, h, 1e-6, st)
    assert all(torch.equal(x, y) for x, y in zip(got, want, strict=True))
    # backward: with and without the residual's gradient, with and without the gain's, added to and written
    x, rstd = want[0], want[2]
    slots = int(_lib.load().spx_rmsnorm_bwd_slots(rows, h))
    for res, train, acc in ((None, True, 0), (dres, True, 1), (dres, False, 0)):
        start = r(slots, h)
        dw = [start.clone() if train else None for _ in range(2)]
        dx = [torch.empty_like(a) for _ in range(2)]
        ld = h if res is not None else 0
        if train:
            _lib.call("spx_rmsnorm_bwd_partial", x, h, gain, b, h, res, ld, rstd, dx[0], h, dw[0], acc, rows, h, st)
        else:
            _lib.call("spx_add_rmsnorm_bwd", x, h, gain, b, h, res, ld, rstd, dx[0], h, None, None, rows, h, st)
        _lib.call("spx_rmsnorm_bwd_parts", x, h, gain, partial, parts, res, ld, rstd, dx[1], h, dw[1], acc, rows, h, st)
        assert torch.equal(dx[0], dx[1]) and (not train or torch.equal(dw[0], dw[1]))


# cut forward and backward products, one on whole tiles, one on the 256 x 256 kernel
@pytest.mark.parametrize("form,m,n,k", [(0, 512, 2048, 8192), (1, 512, 2048, 16384), (0, 333, 2048, 8192), (0, 512, 2048, 512),
                                        (0, 4096, 4096, 4096)])
def test_a_product_leaves_its_parts(form, m, n, k):
    from speculators_amd import _lib

    g = torch.Generator(device="cuda").manual_seed(n + k)
    a = torch.randn(m, k, device="cuda", generator=g).bfloat16()
    b = torch.randn(*((k, n) if form else (n, k)), device="cuda", generator=g).bfloat16()
    nb = int(_lib.load().spx_gemm_auto_workspace_bytes(form, m, n, k, 8))
    ws = torch.empty(max(nb, 16) // 4, device="cuda")
    st, ldb = _lib.stream_ptr(a.device), b.stride(0)
    want, got = (torch.full((m, n), 7.0, device="cuda", dtype=torch.bfloat16) for _ in range(2))
    parts = ctypes.c_int32(0)
    _lib.call("spx_gemm_bf16_auto", form, a, k, b, ldb, want, n, m, n, k, None, 8, ws, ws.nbytes, st)
    _lib.call("spx_gemm_bf16_auto_parts", form, a, k, b, ldb, got, n, m, n, k, 8, ws, ws.nbytes, ctypes.addressof(parts), st)
    assert (parts.value > 1) == (m <= 512 and k >= 8192)
    if parts.value > 1:
        assert bool((got == 7.0).all())  # (not written)
        total = torch.zeros(m, n, device="cuda")
        for p in ws[:parts.value * m * n].view(parts.value, m, n):
            total += p
        got = total.bfloat16()
    assert torch.equal(got, want)
