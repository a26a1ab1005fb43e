// The tile shapes of the deep-ring kernel (gemm_tile_ring.hpp) and its launchers, one per operand type.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

#include "ring_index.hpp"

namespace ptoamd {

struct TileGemmParams;

// id, BM, BN, then waves along M, N, K, stage bytes per row and stages in the ring -- of the plain types and of the
// block-scaled ones, whose matrix instruction takes 128 bytes (fp8) of K --, then waves that only copy, pipelined form.
// Stage widths: 1 KiB where K is split over eight waves of a narrow tile (a copy is then one contiguous KiB of a weight
// row), 256 bytes where it is split over two or the tile is small, one 128-byte slab otherwise.  Block-scaled types split K in
// the first three shapes only.  Ring depth: what 160 KiB hold.  The narrow
// tiles wait for memory whoever copies, so all their waves do; in the others four extra waves only copy, because a wave
// that issues copies stands still while the CU's memory queue is full (128 x 128, bf16 2048 x 2048 x 4096: 50 us with every
// wave copying and multiplying, 33 us with the roles split).  From 64 x 64 on four waves multiply: eight on half of their wave
// tiles read half as much again from LDS per product.  Four against eight, over full grids and part-filled ones: 64 x 64 0.92 to 0.99,
// 96 x 64 and 128 x 64 fp8 0.93 and 0.98, plain types there level, 128 x 128 level, W8A8 on it 0.93, MXFP8 1.02 up
// to K 640 and 0.9 to 1 beyond; 256 x 128 0.94 to 0.98 on a full grid and with one-byte results, and level on a part-filled one and over few
// slabs with 16- or 32-bit results, whose last stage and drain have nothing beside them (bf16 512 x 1024 x 1024 16.0 and 16.2 us).
#define PTOAMD_RING_SHAPES_ALL(X)                                 \
    X(0, 32, 16, 1, 1, 8, 1024, 3, 1, 1, 8, 1024, 3, 0, false)    \
    X(1, 32, 32, 1, 1, 8, 512, 4, 1, 2, 4, 512, 4, 0, false)      \
    X(2, 64, 32, 1, 1, 8, 512, 3, 2, 1, 4, 512, 3, 0, false)      \
    X(3, 64, 64, 2, 1, 2, 256, 4, 2, 2, 1, 256, 4, 4, true)       \
    X(4, 96, 64, 2, 1, 2, 256, 4, 2, 2, 1, 256, 3, 4, true)       \
    X(5, 128, 64, 2, 1, 2, 256, 3, 2, 2, 1, 256, 3, 4, true)      \
    X(6, 128, 128, 2, 2, 1, 128, 4, 2, 2, 1, 128, 4, 4, true)
// the plain types only (the block-scaled columns are empty)
#define PTOAMD_RING_SHAPES_PLAIN(X)                               \
    X(7, 192, 128, 2, 2, 1, 128, 4, 0, 0, 0, 0, 0, 4, true)       \
    X(8, 256, 128, 2, 2, 1, 128, 3, 0, 0, 0, 0, 0, 4, true)
constexpr int RING_SHAPES = 9, RING_SHAPES_SCALED = 7, RING_MAX_STAGE_BYTES = 1024, RING_SHAPE_128X128 = 6;
// Added to the id of a shape with copying waves (3 and up) of the plain types: the form for rows that start on any byte.  So has the
// 32 x 32 shape, as four waves that multiply and four that copy.
constexpr int RING_UNALIGNED = 16, RING_FIRST_UNALIGNED = 3, RING_NARROW_UNALIGNED = 1;
constexpr bool ring_unaligned_shape(int shape) { return shape >= RING_FIRST_UNALIGNED || shape == RING_NARROW_UNALIGNED; }

inline void ring_shape(int shape, int* bm, int* bn)
{
    static const int dims[RING_SHAPES][2] = {
#define PTOAMD_RING_DIM(id, bm, bn, ...) {bm, bn},
        PTOAMD_RING_SHAPES_ALL(PTOAMD_RING_DIM) PTOAMD_RING_SHAPES_PLAIN(PTOAMD_RING_DIM)
#undef PTOAMD_RING_DIM
    };
    *bm = dims[shape % RING_UNALIGNED][0];
    *bn = dims[shape % RING_UNALIGNED][1];
}

// Rows that start on 16 bytes but not all on 128: a stage's 128 bytes of a row lie across two lines, and a copy costs the lines it
// touches.  The shapes with four stages in the ring then copy whole lines (SKEW), from six stages of K on: with fewer the stage more
// that has to land before the first product costs as much (bf16 423 x 1600 x 328 on 64 x 64 tiles 4.8 us, by lines 5.3; 187 x 4502 x
// 248 5.2 and 5.6).  500 sizes (m 33 .. 4096, n 256 .. 8192), by lines against not: 192 x 128 tiles 0.83, 128 x 128 0.80, 96 x 64 0.88, 64 x
// 64 0.92 from 2 KiB of K on, and 0.92 to 0.97 where half of the rows start on a line (pitches of 64 bytes).
inline bool rows_off_lines(const void* a, const void* b, int m, int n, int k_bytes, long lda_bytes, long ldb_bytes, int stage_bytes)
{
    if (k_bytes < 6 * stage_bytes)
        return false;
    const uint64_t last = std::max((uint64_t)(m - 1) * (uint64_t)lda_bytes, (uint64_t)(n - 1) * (uint64_t)ldb_bytes) + (uint64_t)k_bytes;
    if (last + 1024 > UINT32_MAX)  // (lane offsets of whole lines reach a little past a row's)
        return false;
    const uint64_t bits = reinterpret_cast<uintptr_t>(a) | reinterpret_cast<uintptr_t>(b) | (uint64_t)lda_bytes | (uint64_t)ldb_bytes;
    return bits % 16 == 0 && bits % 128 != 0;
}
constexpr int RING_LINES_DEPTH = 4;
// whether a launch of a shape takes that form (plain types, B column-major)
inline bool ring_by_lines(int shape, const void* a, const void* b, int m, int n, int k_bytes, long lda_bytes, long ldb_bytes)
{
    static const struct {
        int stage_bytes, depth;
        bool pipelined;
    } forms[RING_SHAPES] = {
#define PTOAMD_RING_FORM(id, bm, bn, wm, wn, wk, sb, r, swm, swn, swk, ssb, sr, lw, pipe) {sb, r, pipe},
        PTOAMD_RING_SHAPES_ALL(PTOAMD_RING_FORM) PTOAMD_RING_SHAPES_PLAIN(PTOAMD_RING_FORM)
#undef PTOAMD_RING_FORM
    };
    return shape >= 0 && shape < RING_SHAPES && forms[shape].pipelined && forms[shape].depth >= RING_LINES_DEPTH &&
           rows_off_lines(a, b, m, n, k_bytes, lda_bytes, ldb_bytes, forms[shape].stage_bytes);
}

// shape: 0 .. RING_SHAPES - 1, RING_UNALIGNED + one of those of ring_unaligned_shape(), or TILE_PREPARE_ALL
hipError_t launch_gemm_ring_bf16(int shape, const TileGemmParams& p, hipStream_t stream);
hipError_t launch_gemm_ring_f16(int shape, const TileGemmParams& p, hipStream_t stream);
hipError_t launch_gemm_ring_i8(int shape, const TileGemmParams& p, hipStream_t stream);
hipError_t launch_gemm_ring_fp8_e4e4(int shape, const TileGemmParams& p, hipStream_t stream);
hipError_t launch_gemm_ring_fp8_e4e5(int shape, const TileGemmParams& p, hipStream_t stream);
hipError_t launch_gemm_ring_fp8_e5e4(int shape, const TileGemmParams& p, hipStream_t stream);
hipError_t launch_gemm_ring_fp8_e5e5(int shape, const TileGemmParams& p, hipStream_t stream);
hipError_t launch_gemm_ring_fp4(int shape, const TileGemmParams& p, hipStream_t stream);

}  // namespace ptoamd
