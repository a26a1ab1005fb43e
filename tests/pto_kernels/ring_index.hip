// The index arithmetic that the deep-ring kernel's host and device code share, for tests on the host.
#include "gemm_ring.hpp"
#include "gemm_tile_ring.hpp"

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

// A row-major B, the form for rows on any element of shape `shape`: what every lane of every copy of a stage fetches, four numbers each -- row and
// chunk of the stage, matrix row counted from the stage's base row, byte of it; returns how many of them.  *base: that base row.
template <class Cfg>
static int row_copies(int n, int n0, int k, int stage, int most, int* out, int* base)
{
    using Copies = RingRowCopies<Cfg>;
    int count = 0;
    *base = Copies::base(stage);
    for (int lw = 0; lw < Cfg::NW; ++lw)
        for (int q = 0; q < Cfg::NPW; ++q)
            for (int lane = 0; lane < 64 && q * Cfg::NW >= Cfg::A_PIECES; ++lane, ++count) {
                const int row = Copies::row(lw, q, lane), chunk = Copies::chunk(row, lane);
                const int here[4] = {row, chunk, Copies::source(k, stage * Cfg::KR + row) - *base, Copies::byte(n, n0, chunk)};
                for (int i = 0; i < 4 && count < most; ++i)
                    out[4 * count + i] = here[i];
            }
    return count;
}

// *rows, *columns: k rows and columns of a stage
extern "C" int ring_index_row_copies(int shape, int n, int n0, int k, int stage, int most, int* out, int* base, int* rows, int* columns)
{
    switch (shape) {
#define PTOAMD_RING_CASE(id, bm, bn, wm, wn, wk, sb, r, swm, swn, swk, ssb, sr, lw, pipe)                                                 \
    case id:                                                                                                                             \
        if constexpr (ring_unaligned_shape(id)) {                                                                                        \
            using Cfg = std::conditional_t<pipe, RingCfg<bm, bn, wm, wn, wk, sb, r, lw, true, OpBF16x16, true, true>,                    \
                                           RingCfg<bm, bn, 1, 1, 4, sb, r, 4, true, OpBF16x16, true, true>>;                             \
            *rows = Cfg::KR;                                                                                                             \
            *columns = Cfg::BN;                                                                                                          \
            return row_copies<Cfg>(n, n0, k, stage, most, out, base);                                                                    \
        }                                                                                                                                \
        break;
        PTOAMD_RING_SHAPES_ALL(PTOAMD_RING_CASE)
        PTOAMD_RING_SHAPES_PLAIN(PTOAMD_RING_CASE)
#undef PTOAMD_RING_CASE
    }
    return -1;
}
