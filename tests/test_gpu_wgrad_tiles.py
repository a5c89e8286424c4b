"""Weight gradients of few large tiles (spx_gemm_bf16_tn_auto): every tile the choice can fall on, plain and with the
contraction in parts, at ragged results and contractions that end inside a slab or a part."""

import pytest
import torch

pytestmark = pytest.mark.gpu

# (rows, M, N): (tile, in parts); 0: 256 x 256, 1: 128 x 128 by eight waves, 2: 256 x 128, 3: 64 x 128, 4: 128 x 128 by four
CHOICE = {
    (1537, 2056, 2040): (4, False), (2665, 3080, 2048): (2, False), (889, 1032, 2048): (3, False),
    (1777, 2048, 10248): (2, False), (513, 4096, 4096): (0, False), (64, 8, 8): (3, False), (1, 136, 264): (3, False),
    (831, 2664, 1288): (1, False), (5003, 520, 512): (3, True), (8191, 264, 136): (3, True), (20000, 8, 1024): (3, True),
    (14337, 1024, 2056): (2, True), (11935, 1608, 32): (1, True), (4674, 4176, 8): (4, True)}
SHAPES = list(CHOICE)


@pytest.mark.parametrize("t,m,n", SHAPES)
@pytest.mark.parametrize("fp32", [False, True])
@pytest.mark.parametrize("pad", [0, 8])
def test_weight_gradient_against_float64(t, m, n, fp32, pad):
    from speculators_amd.gemm import gemm_tn

    g = torch.Generator(device="cuda").manual_seed(t + m)
    a = torch.randn(t, m + pad, device="cuda", generator=g).bfloat16()[:, :m]
    b = torch.randn(t, n + pad, device="cuda", generator=g).bfloat16()[:, :n]
    want = a.double().t() @ b.double()
    dt = torch.float32 if fp32 else torch.bfloat16
    # (fp32 sums of t products; one rounding to bf16)
    tol = (2e-6 * t ** 0.5 if fp32 else 2 ** -8) * want.abs().max().item() + 1e-4
    got = gemm_tn(a, b, out_dtype=dt)
    assert (got.double() - want).abs().max().item() <= tol
    assert torch.equal(got, gemm_tn(a, b, out_dtype=dt))
    held = torch.full((m, n + 8), 2.0, dtype=dt, device="cuda")
    gemm_tn(a, b, held[:, :n], accumulate=True)
    assert (held[:, :n].double() - want - 2).abs().max().item() <= 2 * tol
    assert (held[:, n:] == 2).all()
    gemm_tn(a, b, held[:, :n])
    assert torch.equal(held[:, :n], got) or (held[:, :n].double() - want).abs().max().item() <= tol


def test_the_choice_falls_on_every_tile():
    from speculators_amd import _lib
    from speculators_amd.gemm import _split_bands

    assert {(t, m, n): (_lib.load().spx_gemm_tn_tile(m, n, t), _split_bands(t, m, n) > 1) for t, m, n in SHAPES} == CHOICE
    assert set(CHOICE.values()) == {(0, False)} | {(tile, parts) for tile in (1, 2, 3, 4) for parts in (False, True)}


def test_workspace_rules():
    from speculators_amd import _lib

    a = torch.zeros(5000, 512, dtype=torch.bfloat16, device="cuda")
    c = torch.zeros(512, 512, device="cuda")
    need = _lib.load().spx_gemm_tn_workspace_bytes(512, 512, 5000)
    assert need == _lib.load().spx_gemm_tn_parts(512, 512, 5000) * 512 * 512 * 4
    ws = torch.zeros(need // 4, device="cuda")
    st = _lib.stream_ptr(a.device)
    args = (a, 512, a, 512, c, 512, 512, 512, 5000, 1, 0)
    _lib.call("spx_gemm_bf16_tn_auto", *args, ws, need, st)
    _lib.call("spx_gemm_bf16_tn_auto", *args, None, 0, st)  # no workspace: never cut
    with pytest.raises(_lib.SpxError):
        _lib.call("spx_gemm_bf16_tn_auto", *args, ws, need - 4, st)
