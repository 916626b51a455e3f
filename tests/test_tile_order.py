"""Row tiles against their definition, row by row: classes in order, rows in index order inside a class."""
import numpy as np
import pytest

from georefine_amd import _fused

NONE = 0xFFFFFFFF


@pytest.mark.parametrize("seed", range(40))
def test_tiles_hold_every_row_once_in_order(seed):
    rng = np.random.default_rng(seed)
    nr, rows = int(rng.integers(1, 17)), int(rng.integers(1, 500))
    row_class = rng.choice(nr, rows, p=rng.dirichlet(np.ones(nr) * rng.choice([0.1, 1, 10]))).astype(np.uint8)
    r, unit, slots, most = (int(rng.integers(1, n)) for n in (40, 17, 300, 200))
    counts = np.bincount(row_class, minlength=nr)
    made = [(*_fused.build_tiles(row_class, nr, r), r)]
    even = _fused.build_balanced_tiles(row_class, nr, unit, slots, most)
    live = int((counts > 0).sum())
    if even is None:
        share = max(-(-int(c) // unit) for c in counts) * unit
        assert live > slots or share > most  # (more slots than classes may still be too few for `most` rows a tile)
    else:
        made.append(even)
        assert even[2] <= most and even[2] % unit == 0 and len(even[1]) <= slots
    for tile_rows, tile_class, height in made:
        assert tile_rows.dtype == np.uint32 and tile_class.dtype == np.uint8
        tiles = tile_rows.reshape(len(tile_class), height)
        assert np.array_equal(np.sort(tile_class), tile_class)
        for c in range(nr):
            of_class = tiles[tile_class == c]
            assert np.array_equal(of_class[of_class != NONE], np.flatnonzero(row_class == c))
        held = (tiles != NONE).sum(axis=1)
        assert np.all(held > 0) and all(np.all(t[:h] != NONE) for t, h in zip(tiles, held))
