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


# the 256 x 256 kernel: last rounds of 16 tiles behind a whole one, of 160, of one, with room for all, some and no parts
@pytest.mark.parametrize("n", [4096, 4100])
@pytest.mark.parametrize("live", [0, 1, 2500, 4097, 4999])
def test_last_round_of_live_tiles_against_float64(n, live):
    from speculators_amd import _lib

    m, k = 5000, 4104
    assert _lib.load().spx_gemm_auto_tile(2, m, n, k, 4) == 0
    g = torch.Generator(device="cuda").manual_seed(live)
    a = torch.randn(m, k, device="cuda", generator=g).bfloat16()
    b = torch.randn(n, k, device="cuda", generator=g).bfloat16()
    weight = torch.rand(m, device="cuda", generator=g) + 0.5
    want = (a[:live].double() @ b.double().t()) * weight[:live].double().unsqueeze(1)
    bound = 2 ** -8 * torch.exp2(want.abs().clamp_min(1e-30).log2().floor())
    bound = bound + 2 ** -22 * (a[:live].double().abs() @ b.double().abs().t()) * weight[:live].double().unsqueeze(1)
    order = torch.arange(m, device="cuda", dtype=torch.int32)
    count = torch.tensor([live], dtype=torch.int32, device="cuda")
    for room in (1024, 100, 0):
        ws = torch.full((room * 65536 + 1024,), 3.0, device="cuda")
        for _ in range(2):
            c = torch.full((m, n + 8), 2.0, dtype=torch.bfloat16, device="cuda")
            _lib.call("spx_gemm_bf16_rows_graded", a, k, b, k, c, n + 8, m, n, k, count, order, weight,
                      torch.ones((), device="cuda"), 1.0, 4, 8, ws if room else None, room * 65536 * 4,
                      _lib.stream_ptr(a.device))
            assert (ws[room * 65536:] == 3).all() and (c[live:] == 2).all() and (c[:, n:] == 2).all()
            assert live == 0 or ((c[:live, :n].double() - want).abs() <= bound).all()


# the 256 x 256 kernel (partial results a whole tile each), and the smaller tiles ([parts][whole tile rows][N])
@pytest.mark.parametrize("m,n,k", [(5000, 4096, 4104), (1300, 2048, 8192), (513, 2048, 4096), (96, 64, 4096)])
def test_device_and_host_find_the_same_parts(m, n, k):
    from speculators_amd import _lib

    lib = _lib.load()
    tile = lib.spx_gemm_auto_tile(2, m, n, k, 4)
    tm, tn = {0: (256, 256), 1: (128, 128), 2: (256, 128), 3: (64, 128)}[tile]
    nbytes = lib.spx_gemm_auto_workspace_bytes(2, m, n, k, 4) if tile else 1024 << 18
    a, b = torch.ones(m, k, device="cuda").bfloat16(), torch.ones(n, k, device="cuda").bfloat16()
    order, weight = torch.arange(m, device="cuda", dtype=torch.int32), torch.ones(m, device="cuda")
    found = set()
    for live in sorted({1, tm, tm + 1, m // 3, m // 2, 2 * m // 3, m - 1, m}):
        count = torch.tensor([live], dtype=torch.int32, device="cuda")
        ws, c = torch.full((nbytes // 4,), 3.0, device="cuda"), torch.empty(m, n, dtype=torch.bfloat16, device="cuda")
        _lib.call("spx_gemm_bf16_rows_graded", a, k, b, k, c, n, m, n, k, count, order, weight, torch.ones((), device="cuda"), 1.0,
                  4, 8, ws, nbytes, _lib.stream_ptr(a.device))
        parts = lib.spx_gemm_graded_parts(m, n, k, 4, 8, nbytes, live)
        tile_rows = -(-live // tm)
        one = tile_rows * -(-n // tn) % 256 * 65536 if tile == 0 else tile_rows * tm * n  # floats of one part
        written = (ws != 3).nonzero()
        assert (c[:live] == torch.tensor(float(k)).bfloat16().item()).all()
        if parts == 1:
            assert len(written) == 0
        else:
            assert (parts - 1) * one <= int(written[-1]) < parts * one
        found.add(parts)
    assert max(found) > 1  # (96 rows are cut in ten whatever counts)
