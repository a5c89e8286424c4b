"""The parts of the graded live-row product (``gemm.rows_graded``): the rule in exact arithmetic, and what the host hands over."""

import os
import subprocess
import sys

import pytest
import torch

from speculators_amd import _lib, gemm


@pytest.fixture
def calls(monkeypatch):
    """``rows_graded`` of ``(M, N, K)`` on the host with the launch replaced: the parts and the workspace's bytes."""
    seen = {}
    monkeypatch.setattr(gemm._lib, "call", lambda name, *a: seen.update({name: a}))
    monkeypatch.setattr(gemm._lib, "stream_ptr", lambda device: 0)
    monkeypatch.setattr(gemm, "_workspaces", gemm._Workspaces())
    count, rows = torch.zeros(1, dtype=torch.int32), torch.zeros(40000, dtype=torch.int32)

    def run(m, n, k):
        a = torch.empty(m, 1, dtype=torch.bfloat16).expand(m, k)
        b = torch.empty(k, dtype=torch.bfloat16).expand(n, k)
        gemm.rows_graded(a, b, count, rows, torch.zeros(m), torch.ones(()), 1.0)
        *_, parts, ws, nbytes, _stream = seen["spx_gemm_bf16_rows_graded"]
        assert ws is None or ws.numel() * 4 >= nbytes
        return parts, nbytes

    return run


@pytest.mark.parametrize("m,n,k", [(4096, 1024, 8192), (888, 2048, 32000), (5000, 512, 56)])
def test_workspace_is_the_one_asked_for(calls, m, n, k):
    alone = calls(m, n, k)
    gemm._split_workspace(torch.device("cpu"), 2 * alone[1] // 4 + 65536)  # left behind by a larger product
    assert calls(m, n, k) == alone



@pytest.mark.parametrize("split,parts", [(None, 8), (1, 1), (2, 2), (3, 3), (4, 4), (8, 8)])
def test_parts_are_bounded_by_the_variable(split, parts):
    env = {k: v for k, v in os.environ.items() if k != "SPX_GEMM_SPLIT_PARTS"}
    if split is not None:
        env["SPX_GEMM_SPLIT_PARTS"] = str(split)
    run = [sys.executable, "-c", "from speculators_amd import gemm; print(gemm.LIVE_TAIL_PARTS if gemm.SPLIT_PARTS > 1 else 1)"]
    assert int(subprocess.run(run, env=env, check=True, capture_output=True, text=True).stdout) == parts


def _rounds(wgs, slabs, cus=256):
    last = wgs % cus
    return slabs * (wgs // cus * 1410 * cus + (1180 * cus + 230 * last if last else 0))


def _last_round(tiles, slabs, max_parts, room, cus=256):
    """Parts of the tiles of the last round: the fewest nanoseconds, each further part 3 % less."""
    rem, parts = tiles % cus, 1
    best = _rounds(rem, slabs) + 6900 * cus
    for p in range(2, max_parts + 1):
        if rem == 0 or slabs // p < 16 or rem * p > room:
            break
        t = _rounds(rem * p, -(-slabs // p)) + cus * (16000 * -(-rem * p // cus) + 4100 + rem * p * 135 // 2)
        if t * 100 < best * 97:
            best, parts = t, p
    return parts


def _small_tiles(tiles, results, slabs, s0, s1, cap):
    """Parts of a product on the smaller tiles: the fewest nanoseconds of those that fit the chip at once."""
    def ns(n):
        return (s0 * cap + s1 * min(tiles * n, cap)) * -(-slabs // n) + (cap * (4100 + n * results * 103 // 100000) if n > 1 else 0)

    fit = [n for n in range(1, min(12, slabs // 6) + 1) if n == 1 or tiles * n <= cap]
    return min(fit, key=ns) if tiles else 1


@pytest.mark.parametrize("m,n,k", [(9003, 4096, 32000), (32760, 2048, 151936), (70000, 256, 4104)])
@pytest.mark.parametrize("room", [0, 100, 1024, 2040])
@pytest.mark.parametrize("split", [1, 3, 8])
def test_parts_of_the_last_round(m, n, k, room, split):
    lib = _lib.load()
    assert lib.spx_gemm_auto_tile(2, m, n, k, 4) == 0
    for tile_rows in range(-(-m // 256) + 1):
        want = _last_round(tile_rows * -(-n // 256), -(-k // 64), split, room if split > 1 else 0)
        for live in {max(0, tile_rows * 256 - 255), tile_rows * 256}:
            assert lib.spx_gemm_graded_parts(m, n, k, 4, split, room * 262144, live) == want, live


TILES = {1: (128, 128, 1, 350, 140), 2: (256, 128, 1, 520, 250), 3: (64, 128, 2, 180, 420)}  # rows, columns, per unit, ns


@pytest.mark.parametrize("tile,m,n,k", [(1, 513, 2048, 4096), (2, 1300, 2048, 8192), (3, 96, 64, 4096), (2, 1536, 2048, 32000)])
def test_parts_on_the_smaller_tiles(tile, m, n, k):
    lib = _lib.load()
    assert lib.spx_gemm_auto_tile(2, m, n, k, 4) == tile
    tm, tn, per, s0, s1 = TILES[tile]
    nbytes = lib.spx_gemm_auto_workspace_bytes(2, m, n, k, 4)
    for live in [0, 1, *range(tm - 1, m, tm), *range(tm, m, tm), m]:
        want = _small_tiles(-(-live // tm) * -(-n // tn), live * n, -(-k // 64), s0, s1, 256 * per)
        assert lib.spx_gemm_graded_parts(m, n, k, 4, 8, nbytes, live) == want, live


# as many partial tiles as the plan asks for at any number of rows: few rows, whole rounds only, every last round there is
@pytest.mark.parametrize("m,n,k", [(3001, 4096, 32000), (9003, 4096, 32000), (32760, 2048, 151936), (70000, 256, 4104),
                                   (5000, 65536, 8192), (5000, 8192, 56)])
@pytest.mark.parametrize("split", [1, 3, 8])
def test_workspace_holds_the_parts_of_any_row_count(m, n, k, split):
    lib = _lib.load()
    assert lib.spx_gemm_auto_tile(2, m, n, k, 4) == 0
    most = 0
    for tile_rows in range(1, -(-m // 256) + 1):
        tiles = tile_rows * -(-n // 256)
        parts = _last_round(tiles, -(-k // 64), split, 256 * 8)
        most = max(most, tiles % 256 * parts if parts > 1 else 0)
    nbytes = lib.spx_gemm_graded_workspace_bytes(m, n, k, 4, split)
    assert nbytes == most * 262144
    assert gemm._graded_workspace(m, n, k, 4, split) * 4 == nbytes
