// The index arithmetic that the deep-ring kernel's host and device code share, for tests on the host.
#include "ring_index.hpp"

using namespace ptoamd;

extern "C" int ring_index_group() { return RING_GROUP; }

// tiles of bm x bn over m x n: the tile of every workgroup, rows and columns one after the other; returns the number of workgroups
extern "C" int ring_index_tiles(int m, int n, int bm, int bn, int group_m, int most, int* rows, int* columns)
{
    const RingTiles t = ring_tiles(m, n, bm, bn, group_m);
    for (int block = 0; block < t.grid && block < most; ++block) {
        const RingTile at = t.tile(block);
        rows[block] = at.row;
        columns[block] = at.column;
    }
    return t.grid;
}
