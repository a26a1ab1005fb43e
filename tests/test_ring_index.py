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


@pytest.mark.parametrize("shape", [1, 3, 4, 5, 6, 7, 8])
def test_copies_of_a_row_major_b_stay_inside_it(index, shape):
    """Every 16 bytes that a copying lane fetches lie in one k row of B, in each stage of every K from one chunk of eight rows on and each
    tile column of every N from one chunk of columns on; they hold the row and the columns that are multiplied there, and the 32-bit offsets
    reach no more rows than the launcher allows for."""
    most = 64 * 1024
    out, one = np.empty((most, 4), np.int32), [ctypes.c_int() for _ in range(3)]

    def copies(n, n0, k, stage):
        count = index.ring_index_row_copies(shape, n, n0, k, stage, most, out.ctypes.data_as(ctypes.c_void_p), *(ctypes.byref(x) for x in one))
        assert 0 < count <= most
        return out[:count].T.astype(np.int64), one[0].value
    copies(64, 0, 64, 0)
    rows, columns = one[1].value, one[2].value
    ns = list(range(8, 25)) + [columns - 1, columns, columns + 1, columns + 7, columns + 8, 3 * columns - 3]
    ks = list(range(8, 25)) + [rows - 1, rows, rows + 1, rows + 7, rows + 8, 2 * rows + 13, 5 * rows + 6]
    for n in ns:
        for k in ks:
            for n0 in range(0, n, columns):
                for stage in range((k + rows - 1) // rows):
                    (row, chunk, src, byte), base = copies(n, n0, k, stage)
                    assert len(set(zip(row, chunk))) == row.size == rows * columns // 8 and row.min() == 0 and row.max() == rows - 1 and chunk.min() == 0 and chunk.max() == columns // 8 - 1
                    assert src.min() >= 0 and src.max() < 1024 // 2 + 8 and base >= 0 and (base + src).max() < k, (n, k, n0, stage)
                    assert byte.min() >= 0 and byte.max() + 16 <= 2 * n, (n, k, n0, stage)
                    r = stage * rows + row
                    whole = (r | 7) < k
                    assert np.array_equal((base + src)[whole], r[whole])
                    # the eight rows that K ends in: the last eight, so that a row of them stands k - 8 further on than its place in its chunk
                    ends = ~whole & (r < k)
                    assert np.array_equal((base + src)[ends], (k - 8 + (r & 7))[ends])
                    wanted = n0 * 2 + chunk * 16  # first byte of the chunk's columns; what is fetched starts there or, shifted by up to 14 bytes, in front
                    stored = wanted < 2 * n
                    assert ((wanted - byte)[stored] >= 0).all() and ((wanted - byte)[stored] < 16).all() and np.array_equal((wanted - byte)[stored] > 0, (wanted + 16 > 2 * n)[stored])
