"""Index arithmetic of the deep-ring kernel, the code that the kernel runs compiled for the host."""
import ctypes
import os

import numpy as np
import pytest

LIB = os.path.join(os.path.dirname(os.path.abspath(__file__)), "pto_kernels", "build", "libringindex.so")


@pytest.fixture(scope="module")
def index():
    assert os.path.exists(LIB), "build the test libraries first: make -C tests/pto_kernels"
    return ctypes.CDLL(LIB)


def _tiles(index, tiles_m, tiles_n, group_m, bm=32, bn=64):
    m, n = tiles_m * bm - 7, tiles_n * bn - 33
    rows, columns = (np.full(tiles_m * tiles_n, -1, np.int32) for _ in range(2))
    grid = index.ring_index_tiles(m, n, bm, bn, group_m, rows.size, rows.ctypes.data_as(ctypes.c_void_p), columns.ctypes.data_as(ctypes.c_void_p))
    assert grid == tiles_m * tiles_n
    return rows, columns


@pytest.mark.parametrize("group_m", [1, 2, 3, 4, 5, 8, 40])
def test_every_tile_once(index, group_m):
    """Whole groups of rows, last groups of one, two and three, all rows in one group, whatever group is asked for."""
    for tiles_m in range(1, 41):
        for tiles_n in (1, 2, 3, 5, 8, 31, 257):
            rows, columns = _tiles(index, tiles_m, tiles_n, group_m)
            assert rows.min() >= 0 and rows.max() < tiles_m and columns.min() >= 0 and columns.max() < tiles_n, (tiles_m, tiles_n)
            assert np.array_equal(np.sort(rows * tiles_n + columns), np.arange(tiles_m * tiles_n)), (tiles_m, tiles_n)


def test_an_xcd_walks_a_run_of_tiles_by_groups_of_rows(index):
    group, tiles_m, tiles_n = index.ring_index_group(), 11, 16
    rows, columns = _tiles(index, tiles_m, tiles_n, group)
    walked = np.concatenate([np.arange(x, rows.size, 8) for x in range(8)])  # workgroups of XCD 0, of XCD 1, ...
    rows, columns = rows[walked], columns[walked]
    ref = [(r, c) for first in range(0, tiles_m, group) for c in range(tiles_n) for r in range(first, min(first + group, tiles_m))]
    assert list(zip(rows, columns)) == ref


def test_divisions_by_products(index):
    """Grids up to many tiles: 16-row panels of large matrices."""
    for tiles_m, tiles_n in ((1, 1 << 17), (1 << 17, 1), (9, 40_009), (4097, 67), (8, 65_537)):
        for group_m in (4, tiles_m if tiles_m <= 8 else 4):
            rows, columns = _tiles(index, tiles_m, tiles_n, group_m)
            assert np.array_equal(np.sort(rows.astype(np.int64) * tiles_n + columns), np.arange(tiles_m * tiles_n)), (tiles_m, tiles_n)
