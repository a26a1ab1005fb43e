// Instantiates gemm_tile_ring_kernel for one operand type at the shapes of gemm_ring.hpp.  Included by
// gemm_ring_<op>.hip with PTOAMD_RING_OP (the traits type) and PTOAMD_RING_FN (the launcher's name) defined.
#include <algorithm>

#include "common_host.hpp"
#include "gemm_ring.hpp"
#include "gemm_tile_ring.hpp"

namespace ptoamd {

template <class Cfg>
static hipError_t launch_ring(const TileGemmParams& p, hipStream_t stream)
{
    const hipError_t e = ensure_dynamic_lds<&gemm_tile_ring_kernel<Cfg>>(Cfg::LDS_BYTES);
    if (e != hipSuccess || p.m <= 0)  // m = 0: only make the kernel ready to launch on the current device
        return e;
    const RingTiles tiles = ring_tiles(p, Cfg::BM, Cfg::BN);
    hipLaunchKernelGGL((gemm_tile_ring_kernel<Cfg>), dim3(tiles.grid), dim3(Cfg::THREADS), Cfg::LDS_BYTES, stream, p, tiles);
    return hipGetLastError();
}

// Rows that start on 16 bytes but not all on 128: a stage's 128 bytes of a row lie across two lines, and a copy costs the lines it
// touches.  The shapes with four stages in the ring then copy whole lines (SKEW), from six stages of K on: with fewer the stage more
// that has to land before the first product costs as much (bf16 423 x 1600 x 328 on 64 x 64 tiles 4.8 us, by lines 5.3; 187 x 4502 x
// 248 5.2 and 5.6).  500 sizes (m 33 .. 4096, n 256 .. 8192), by lines against not: 192 x 128 tiles 0.83, 128 x 128 0.80, 96 x 64 0.88, 64 x
// 64 0.92 from 2 KiB of K on, and 0.92 to 0.97 where half of the rows start on a line (pitches of 64 bytes).
static bool rows_off_lines(const TileGemmParams& p, int stage_bytes)
{
    if (p.k_bytes < 6 * stage_bytes)
        return false;
    const uint64_t last = std::max((uint64_t)(p.m - 1) * (uint64_t)p.lda_bytes, (uint64_t)(p.n - 1) * (uint64_t)p.ldb_bytes) + (uint64_t)p.k_bytes;
    if (last + 1024 > UINT32_MAX)  // (lane offsets of whole lines reach a little past a row's)
        return false;
    const uint64_t bits = reinterpret_cast<uintptr_t>(p.a) | reinterpret_cast<uintptr_t>(p.b) | (uint64_t)p.lda_bytes | (uint64_t)p.ldb_bytes;
    return bits % 16 == 0 && bits % 128 != 0;
}

template <bool BND, int BM, int BN, int WM, int WN, int WK, int SB, int R, int LW, bool PIPE, class Op>
static hipError_t launch_ring_plain(const TileGemmParams& p, hipStream_t stream)
{
    if constexpr (!BND && PIPE && R >= 4) {
        using Skewed = RingCfg<BM, BN, WM, WN, WK, SB, R, LW, PIPE, Op, false, false, true>;
        if (p.m <= 0) {  // (both forms are made ready)
            const hipError_t e = launch_ring<Skewed>(p, stream);
            if (e != hipSuccess)
                return e;
        } else if (rows_off_lines(p, SB)) {
            return launch_ring<Skewed>(p, stream);
        }
    }
    return launch_ring<RingCfg<BM, BN, WM, WN, WK, SB, R, LW, PIPE, Op, BND>>(p, stream);
}

template <class Op, bool BND = false>
static hipError_t launch_ring_shape(int shape, const TileGemmParams& p, hipStream_t stream)
{
    switch (shape) {
#define PTOAMD_RING_CASE(id, bm, bn, wm, wn, wk, sb, r, swm, swn, swk, ssb, sr, lw, pipe)                            \
    case id:                                                                                                        \
        if constexpr (Op::SCALED)                                                                                   \
            return launch_ring<RingCfg<bm, bn, swm, swn, swk, ssb, sr, lw, pipe, Op>>(p, stream);                   \
        else                                                                                                        \
            return launch_ring_plain<BND, bm, bn, wm, wn, wk, sb, r, lw, pipe, Op>(p, stream);
        PTOAMD_RING_SHAPES_ALL(PTOAMD_RING_CASE)
#undef PTOAMD_RING_CASE
        default: break;
    }
    if constexpr (!Op::SCALED) {
        switch (shape) {
#define PTOAMD_RING_CASE(id, bm, bn, wm, wn, wk, sb, r, swm, swn, swk, ssb, sr, lw, pipe) \
    case id: return launch_ring_plain<BND, bm, bn, wm, wn, wk, sb, r, lw, pipe, Op>(p, stream);
            PTOAMD_RING_SHAPES_PLAIN(PTOAMD_RING_CASE)
#undef PTOAMD_RING_CASE
            default: break;
        }
    }
    return hipErrorInvalidValue;
}

// the form for rows at any alignment, shapes with copying waves only
template <class Op>
static hipError_t launch_ring_unaligned(int shape, const TileGemmParams& p, hipStream_t stream)
{
    switch (shape) {
#define PTOAMD_RING_CASE(id, bm, bn, wm, wn, wk, sb, r, swm, swn, swk, ssb, sr, lw, pipe)                            \
    case id:                                                                                                        \
        if constexpr (pipe)                                                                                         \
            return launch_ring<RingCfg<bm, bn, wm, wn, wk, sb, r, lw, pipe, Op, false, true>>(p, stream);           \
        break;
        PTOAMD_RING_SHAPES_ALL(PTOAMD_RING_CASE)
        PTOAMD_RING_SHAPES_PLAIN(PTOAMD_RING_CASE)
#undef PTOAMD_RING_CASE
        default: break;
    }
    return hipErrorInvalidValue;
}

hipError_t PTOAMD_RING_FN(int shape, const TileGemmParams& p, hipStream_t stream)
{
#ifdef PTOAMD_RING_BND  // the 16-bit types also take a row-major B
    constexpr bool has_bnd = true;
#else
    constexpr bool has_bnd = false;
#endif
    if (shape >= RING_UNALIGNED && shape != TILE_PREPARE_ALL) {
        if constexpr (!PTOAMD_RING_OP::SCALED)
            if (!p.b_nd)
                return launch_ring_unaligned<PTOAMD_RING_OP>(shape - RING_UNALIGNED, p, stream);
        return hipErrorInvalidValue;
    }
    if (shape != TILE_PREPARE_ALL) {
        if (!p.b_nd)
            return launch_ring_shape<PTOAMD_RING_OP>(shape, p, stream);
        if constexpr (has_bnd)
            return launch_ring_shape<PTOAMD_RING_OP, true>(shape, p, stream);
        return hipErrorInvalidValue;
    }
    const TileGemmParams none{};
    for (int s = 0; s < (PTOAMD_RING_OP::SCALED ? RING_SHAPES_SCALED : RING_SHAPES); ++s) {
        hipError_t e = launch_ring_shape<PTOAMD_RING_OP>(s, none, stream);
        if constexpr (has_bnd) {
            if (e == hipSuccess)
                e = launch_ring_shape<PTOAMD_RING_OP, true>(s, none, stream);
        }
        if constexpr (!PTOAMD_RING_OP::SCALED) {
            if (e == hipSuccess && s >= RING_FIRST_UNALIGNED)
                e = launch_ring_unaligned<PTOAMD_RING_OP>(s, none, stream);
        }
        if (e != hipSuccess)
            return e;
    }
    return hipSuccess;
}

}  // namespace ptoamd
