// Index arithmetic of the deep-ring kernel (gemm_tile_ring.hpp) that host and kernel share.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

namespace ptoamd {

// n / d for 0 <= n < 2^31 as a product (division by an invariant integer through multiplication, Granlund and Montgomery 1994): with l = ceil(log2 d) and magic = ceil(2^(31 + l) / d), which is below 2^32, the error of
// n * magic / 2^(31 + l) is below 1 / d.
struct RingDivisor {
    uint32_t magic, shift;
    __host__ static RingDivisor of(uint32_t d)
    {
        uint32_t l = 0;
        while ((1ull << l) < d)
            ++l;
        return {(uint32_t)(((1ull << (31 + l)) + d - 1) / d), 31 + l};
    }
    __host__ __device__ __forceinline__ int divide(int n) const { return (int)(((uint64_t)(uint32_t)n * magic) >> shift); }
};

struct RingTile {
    int row, column;
};
// Workgroup -> tile, prepared by the host: `grid` tiles in tiles_m rows, walked in groups of rows; per_group tiles make a group of
// RING_GROUP rows (the last one has fewer), or all tiles are one group of tiles_m rows (per_group = grid).  divisor: of per_group,
// or of tiles_m.  Two divisions of run-time values in the kernel took 90 scalar instructions.
constexpr int RING_GROUP = 4;
struct RingTiles {
    int grid, tiles_m, per_group;
    RingDivisor divisor;

    // Workgroup ids go round-robin to the 8 XCDs; XCD x takes a contiguous run of tiles, walked in groups of RING_GROUP tile rows or
    // in one of all rows, so that what an L2 holds is a few panels of A and of B.
    __host__ __device__ __forceinline__ RingTile tile(uint32_t block) const
    {
        const int xcd = block & 7;
        const int lid = xcd * (grid >> 3) + (xcd < (grid & 7) ? xcd : grid & 7) + (int)(block >> 3);
        const int quotient = divisor.divide(lid);
        if (per_group == grid)
            return {lid - quotient * tiles_m, quotient};
        const int in_group = lid - quotient * per_group, first = quotient * RING_GROUP, rows = tiles_m - first < RING_GROUP ? tiles_m - first : RING_GROUP;
        static_assert(RING_GROUP == 4, "the divisions by a group's rows are spelled out");
        const int column = rows == 4 ? in_group >> 2 : rows == 3 ? (int)(uint32_t)(((uint64_t)(uint32_t)in_group * 0xAAAAAAABu) >> 33) : in_group >> (rows - 1);
        return {first + in_group - column * rows, column};
    }
};
// group_m: all rows are one group where it holds them, or where RING_GROUP does
inline RingTiles ring_tiles(int m, int n, int bm, int bn, int group_m)
{
    RingTiles t;
    const int tiles_n = (n + bn - 1) / bn;
    t.tiles_m = (m + bm - 1) / bm;
    t.grid = t.tiles_m * tiles_n;
    const bool one_group = std::max(group_m, RING_GROUP) >= t.tiles_m;
    t.per_group = one_group ? t.grid : RING_GROUP * tiles_n;
    t.divisor = RingDivisor::of(one_group ? t.tiles_m : t.per_group);
    return t;
}

}  // namespace ptoamd
