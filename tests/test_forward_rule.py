"""Which decoder projections run on this library's kernels forward ("mixed"): a rule of sizes alone, no GPU needed."""

import random

import pytest

from speculators_amd import _lib, gemm


@pytest.mark.parametrize("rows,n,k,own", [
    # up to 1024 rows on tiles of 192 rows: 70B q/k/v and gate/up and 8B gate/up stay with the library, short contractions do not
    (777, 10240, 16384, False), (1024, 10240, 16384, False), (1024, 10240, 8192, False), (160, 57344, 8192, False),
    (384, 57344, 8192, False), (260, 28672, 4096, False), (384, 28672, 4096, False), (888, 28672, 4096, False),
    (600, 16384, 2048, True), (768, 16384, 2048, True),
    # two rounds of 192 x 192, a contraction in parts, a cut last round, smaller tiles
    (3001, 6144, 8192, True), (1300, 4096, 14336, True), (4096, 6144, 8192, True), (512, 6144, 8192, True), (1024, 2048, 2048, True)])
def test_measured_products(rows, n, k, own):
    assert gemm._own_forward(rows, n, k) == own


def test_nothing_that_ran_here_without_the_tall_tiles_goes_to_the_library():
    rnd = random.Random(1)
    for _ in range(4000):
        m, n, k = rnd.randint(8, 5000), 8 * rnd.randint(16, 4096), 8 * rnd.randint(64, 2048)
        tile = _lib.load().spx_gemm_auto_tile(2, m, n, k, gemm.TAIL_PARTS)  # the choice without tiles of 192 rows
        if tile and m <= 1024:
            assert gemm._own_forward(m, n, k), (m, n, k)


@pytest.mark.parametrize("rows,n,k,here", [
    # short contractions, a cut last round, long contractions; whole rounds between stay with the library, as do no rows and
    # sizes that workgroups do not walk
    (888, 16384, 2048, True), (32760, 12288, 2048, True), (3001, 28672, 4096, True), (5000, 6144, 16384, True),
    (4096, 28672, 4096, False), (888, 28672, 4096, False), (0, 16384, 2048, False), (3001, 16384, 2080, False),
    (3001, 16380, 2048, False)])
def test_products_that_workgroups_walk(rows, n, k, here):
    assert not gemm._own_forward(rows, n, k) and gemm._walking_forward(rows, n, k) == here
    assert (gemm._forward_route("mixed", gemm.TAIL_PARTS, rows, n, k)[0] != gemm.LINEAR) == here
    assert gemm._forward_route("mixed", gemm.TAIL_PARTS, rows, n, k, False)[0] == gemm.LINEAR


def test_routes_go_by_the_parts_that_are_asked_for(monkeypatch):
    """A route of another number of parts than the running one is the route that runs with that number, whatever was asked first."""
    shapes = [(m, n, k) for m in (300, 1500, 3001, 4096, 5000) for n, k in ((28672, 4096), (6144, 16384), (6144, 8192), (4096, 4096))]

    def forget():
        for f in vars(gemm).values():
            getattr(f, "cache_clear", lambda: None)()

    def routes(parts):
        return [gemm._forward_route("mixed", parts, *s, lines) for s in shapes for lines in (False, True)]

    def walk():
        return [gemm._walking_forward(*s) for s in shapes]

    forget()
    asked, walked = {p: routes(p) for p in (4, 1)}, {}
    for parts in (1, 4):
        monkeypatch.setattr(gemm, "TAIL_PARTS", parts)
        walked[parts] = walk()
        forget()
        assert routes(parts) == asked[parts] and walk() == walked[parts]
    assert asked[1] != asked[4] and walked[1] != walked[4]
    forget()


# (rows, columns, contraction, tile): results of no whole number of 256 columns, where the large tile is not the walking one, and
# of such a number, where it is
@pytest.mark.parametrize("m,n,k,tile", [(1400, 4160, 8192, 2), (8192, 2880, 4096, 2), (700, 2880, 11520, 4),
                                        (1400, 2048, 16384, 5), (8192, 4096, 14336, 5), (3500, 2048, 16384, 5)])
def test_input_gradients_on_large_tiles(m, n, k, tile):
    assert _lib.load().spx_gemm_auto_tile(1, m, n, k, 4) == tile


# a contraction that ends inside a slab, columns that are no multiple of 8, two slabs: no workgroup walks, and the large tile is left; then
# sizes next to them that are walked
@pytest.mark.parametrize("m,n,k,large", [(8288, 2944, 808, False), (2048, 17784, 1336, False), (4352, 4288, 72, False),
                                         (6000, 16384, 128, False), (2048, 17784, 1344, True), (6000, 16384, 192, True)])
def test_large_tiles_that_do_not_walk(m, n, k, large):
    assert (_lib.load().spx_gemm_auto_tile(0, m, n, k, 4) == 0) == large
    if k % 64 == 0:
        assert gemm._walking_forward(m, n, k) == large
