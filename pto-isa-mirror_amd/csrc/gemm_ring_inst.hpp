// Instantiates gemm_tile_ring_kernel for one operand type at the shapes of gemm_ring.hpp.  Included by
// gemm_ring_<op>.hip with PTOAMD_RING_OP (the traits type) and PTOAMD_RING_FN (the launcher's name) defined.
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
    const RingTiles tiles = ring_tiles(p.m, p.n, Cfg::BM, Cfg::BN, p.group_m);
    hipLaunchKernelGGL((gemm_tile_ring_kernel<Cfg>), dim3(tiles.grid), dim3(Cfg::THREADS), Cfg::LDS_BYTES, stream, p.a, p.b, (uint32_t)p.lda_bytes, (uint32_t)p.ldb_bytes, p.m, p.n, p.k_bytes, tiles.grid,
                       tiles.tiles_m, tiles.per_group, tiles.divisor.magic, tiles.divisor.shift, p);
    return hipGetLastError();
}

template <bool BND, int BM, int BN, int WM, int WN, int WK, int SB, int R, int LW, bool PIPE, class Op>
static hipError_t launch_ring_plain(const TileGemmParams& p, hipStream_t stream)
{
    if constexpr (!BND && PIPE && R >= RING_LINES_DEPTH) {
        using Skewed = RingCfg<BM, BN, WM, WN, WK, SB, R, LW, PIPE, Op, false, false, true>;
        if (p.m <= 0) {  // (both forms are made ready)
            const hipError_t e = launch_ring<Skewed>(p, stream);
            if (e != hipSuccess)
                return e;
        } else if (rows_off_lines(p.a, p.b, p.m, p.n, p.k_bytes, p.lda_bytes, p.ldb_bytes, SB)) {
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

// the form for rows at any alignment: shapes with copying waves, and 32 x 32 as four waves that multiply and four that copy
template <class Op, bool BND = false>
static hipError_t launch_ring_unaligned(int shape, const TileGemmParams& p, hipStream_t stream)
{
    switch (shape) {
#define PTOAMD_RING_CASE(id, bm, bn, wm, wn, wk, sb, r, swm, swn, swk, ssb, sr, lw, pipe)                            \
    case id:                                                                                                        \
        if constexpr (pipe)                                                                                         \
            return launch_ring<RingCfg<bm, bn, wm, wn, wk, sb, r, lw, pipe, Op, BND, true>>(p, stream);             \
        else if constexpr (id == RING_NARROW_UNALIGNED)                                                             \
            return launch_ring<RingCfg<bm, bn, 1, 1, 4, sb, r, 4, true, Op, BND, true>>(p, stream);                 \
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
            if (!p.b_nd || has_bnd)
                return p.b_nd ? launch_ring_unaligned<PTOAMD_RING_OP, has_bnd>(shape - RING_UNALIGNED, p, stream)
                              : launch_ring_unaligned<PTOAMD_RING_OP>(shape - RING_UNALIGNED, p, stream);
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
            if (e == hipSuccess && ring_unaligned_shape(s))
                e = launch_ring_unaligned<PTOAMD_RING_OP>(s, none, stream);
            if (e == hipSuccess && has_bnd && ring_unaligned_shape(s))
                e = launch_ring_unaligned<PTOAMD_RING_OP, has_bnd>(s, none, stream);
        }
        if (e != hipSuccess)
            return e;
    }
    return hipSuccess;
}

}  // namespace ptoamd
