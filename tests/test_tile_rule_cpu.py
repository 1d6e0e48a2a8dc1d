"""The default y chunk of the Laplacian step against a sweep of every chunk on the MI355X: one of those within 5 % of
the fastest, for orders 8, 10, 12 and 16 and grids of 48 to 400 planes.  (3 planes at FD16 80^3 take 1.63 times as
long as 7, and 3 planes at 96^3 1.41 times as long as 10.)"""
import pytest

from konglong_amd.batch import Autotuner
from konglong_amd.kernel import KernelCPU

BEST = {  # (ny, nx, nz): chunks for orders 8, 10, 12 and for 16
    (48, 48, 48): ([2], [2]),
    (64, 64, 64): ([2], [2]),
    (80, 80, 80): ([4, 7], [7]),
    (96, 96, 96): ([5], [10]),
    (113, 97, 105): ([6], [13]),
    (128, 128, 128): ([8], [16]),
    (128, 60, 140): ([7, 8], [13]),
    (160, 150, 140): ([20], [40]),
    (200, 200, 200): ([40], [40]),
    (256, 256, 256): ([64], [128]),
    (400, 400, 400): ([37, 40, 45, 50, 58, 67, 80, 100], [67, 80, 100, 200]),
}


@pytest.mark.parametrize("shape", BEST, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("order", [8, 10, 12, 16])
def test_default_chunk_is_near_the_fastest(shape, order):
    ny, nx, nz = shape
    k = KernelCPU(nx, ny, nz, 10.0, 10.0, 10.0, order=order)
    assert k.get_tile()[:2] == (min(64, nz), 8)
    assert k.get_tile()[2] in BEST[shape][order == 16]


@pytest.mark.parametrize("ny", [1, 2, 7, 40, 331, 5000])
@pytest.mark.parametrize("tile", [(0, 0), (16, 16), (64, 4), (8, 64)])
def test_chunk_lies_in_the_grid(ny, tile):
    k = KernelCPU(50, ny, 70, 10.0, 10.0, 10.0)
    k.set_tile(*tile)
    assert 1 <= k.get_tile()[2] <= ny
    k.set_tile(0, 0, 9)
    assert k.get_tile()[2] == 9
    k.set_tile(0, 0, -1)
    assert 1 <= k.get_tile()[2] <= ny


def test_tile_without_room_is_refused():
    """128 z lanes leave 4 x rows in 512 threads, the radius of FD16 is 8: no x tile fits, and looking for one by
    halving never ended."""
    k = KernelCPU(64, 64, 256, 10.0, 10.0, 10.0, order=16)
    before = k.get_tile()
    with pytest.raises(Exception, match="no room"):
        k.set_tile(128)
    assert k.get_tile() == before
    k = KernelCPU(64, 64, 256, 10.0, 10.0, 10.0, order=8)
    k.set_tile(128)
    assert k.get_tile()[:2] == (128, 4)


def test_autotuner_times_no_tile_twice():
    """The first-derivative passes run at most 64 z lanes, so a wider candidate is another one again."""
    seen = [(min(tz, 64), min(tx, 32)) for tz, tx in Autotuner.TILES_FIRST_DERIV]
    assert len(set(seen)) == len(seen)
    assert all(t in Autotuner.TILES_FIRST_DERIV for t in ((64, 8), (64, 4), (32, 8), (16, 16)))
