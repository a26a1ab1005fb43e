// Tiled MFMA GEMM, deep-ring form: for grids that leave CUs idle or have one workgroup per CU, and for few rows of A.
//
// What bounds such a grid is the latency of the copy-in, not the matrix cores and not a bandwidth: the 128 x 128 DMA
// tile takes 0.6 us per 128-byte slab whether 128 or 256 of them run, because only one slab is in flight while one is
// multiplied.  Here a CU's LDS holds a ring of R stages, R - 1 of them in flight, a tile's shape is chosen so that one
// round of workgroups covers the matrix, and a stage of a narrow tile is up to 1 KiB of every row, split over groups of
// waves along K (each group multiplies its own part of the stage; the partial sums meet in LDS when K is done).  With
// 16 columns of B per workgroup a decode step of 4096 columns reads its weights through 256 CUs.
//
//   TLOAD      global_load_lds_dwordx4, lane-linear in LDS, 16-byte chunks swizzled on the global-address side; every wave
//              issues the same number of copies per stage, so a stage is waited for by count (vmcnt)
//   TEXTRACT   ds_read_b128 fragments; the swizzle makes the 16 rows of a lane group fall into different banks
//   TMATMUL    the 16x16 matrix instructions of every operand type (block-scaled types: one dword of E8M0 per 128 K)
//   sync       one workgroup barrier per stage: behind it the stage has landed and the previous one may be overwritten
//   B row-major (BND, 16-bit types): a stage holds its k rows as they lie in memory and ds_read_b64_tr_b16 turns four of them at a
//              time into fragments, so no copy of B is made and no thread moves elements.  Measured, bf16: 2048 x 4096 x 4096
//              57 us (column-major B 56; re-ordered through a workspace first 80; scattered by the register-staged loader
//              101), 24 x 4096 x 4096 14.2 us (column-major 9.6: here a copy takes 32 bytes of each row; loader 58)
//   rows at any alignment (ANY, plain types): LDS-DMA wants dword-aligned addresses, so where rows start on other bytes (an odd
//              number of 16-bit elements) the waves that copy go through registers, unaligned 16-byte loads two or three stages
//              ahead of their ds_write_b128; everything behind the barrier is the same.
//              A stage takes about twice as long as by LDS-DMA.
//              Measured, bf16, against the register-staged tile chosen by grid size: 64 x 4097 x 4095 28 us (63), 1000 x 2049 x 2047
//              33 (57; 2048 x 2048 by LDS-DMA: 17), 2100 x 2049 x 2047 43 (61), 4000 x 1025 x 4097 73 (110)
//              With a row-major B (BND as well) a chunk of B is eight columns of a k row; the chunk that N ends in is the 16 bytes that end
//              there, shifted in registers.  bf16 18 x 308 x 7274 18.9 us (register-staged loader 134), 1111 x 3347 x 4028 54 (194)
//   rows on 16 bytes off the 128-byte lines (SKEW, plain types, shapes with four stages): a copy's cost is the lines it touches, and
//              a stage of such a row lies across two per 128 bytes.  Each row's copies are cut at its lines instead, up to 112 bytes
//              ahead of the row's k, so a stage is multiplied when the next one has landed as well.  bf16 1237 x 4100 x 2056 with
//              bias and relu 32.2 -> 25.6 us, 24.3 where the pitch is a multiple of 128 bytes
//   K tail     copies never read past a row: a chunk that would is read as the 16 bytes that END at the row's end, and the
//              last stage's fragments are masked in registers -- the same bytes of A and B, so k positions still agree
#pragma once
#include <cstddef>

#include "gemm_tile_dtl.hpp"
#include "ring_index.hpp"

namespace ptoamd {

// fp4 E2M1 on the 16x16x128 scaled instruction: a lane holds 16 bytes of one of 16 rows = one MX block, and its scale
struct OpFP4x16 {
    static constexpr int BLK = 16, ACC_REGS = 4;
    using Acc = f32x4;
    using Elem = float;
    static constexpr int FRAG_BYTES = 16;
    static constexpr bool SCALED = true;
    static constexpr int GROUPS_PER_SLAB = 8;
    __device__ static __forceinline__ void mma(Acc& c, const uint4* a, const uint4* b, uint32_t sa, uint32_t sb)
    {
        i32x8 av = {0, 0, 0, 0, 0, 0, 0, 0}, bv = {0, 0, 0, 0, 0, 0, 0, 0};
        av.s0 = a[0].x; av.s1 = a[0].y; av.s2 = a[0].z; av.s3 = a[0].w;
        bv.s0 = b[0].x; bv.s1 = b[0].y; bv.s2 = b[0].z; bv.s3 = b[0].w;
        c = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(bv, av, c, 4, 4, 0, (int)sb, 0, (int)sa);
    }
};

// WM x WN x WK waves: WK groups share the tile and split every stage of SB bytes per row along K; R stages in the ring
template <int BM_, int BN_, int WM_, int WN_, int WK_, int SB_, int R_, int LW_, bool PIPE_, class Op_, bool BND_ = false, bool ANY_ = false, bool SKEW_ = false>
struct RingCfg {
    static constexpr int BM = BM_, BN = BN_, WM = WM_, WN = WN_, WK = WK_, SB = SB_, R = R_;
    static constexpr bool PIPE = PIPE_, BND = BND_, ANY = ANY_, SKEW = SKEW_;  // B is row-major [K][N]; rows start on any byte; on any 16
    using Op = Op_;
    static constexpr int CW = WM * WN * WK, LW = LW_, THREADS = (CW + LW) * 64;
    static constexpr int NW = LW > 0 ? LW : CW;  // waves that copy
    static constexpr int WTM = BM / WM, WTN = BN / WN, MB = WTM / 16, NB = WTN / 16;
    static constexpr int FR = Op::FRAG_BYTES / 16, KB = 4 * Op::FRAG_BYTES;  // bytes of K one matrix instruction takes
    static constexpr int KW = SB / WK, KSTEPS = KW / KB;
    static constexpr int ROWS = BM + BN, CPR = SB / 16, RPP = 1024 / SB;  // chunks per row, rows per 1 KiB piece
    static constexpr int PIECES = ROWS * SB / 1024, A_PIECES = BM * SB / 1024, NPW = PIECES / NW;
    // Block scales, SPS dwords (of four groups each) per row and stage.  A copy's cost is the 128-byte lines it touches, whatever it
    // takes of them: a dword or two per row, as each stage needs them, made them half as expensive as the operands (96 x 64 tile,
    // fp8: 160 lines beside 320 per stage).  Such tiles of 160 rows and more (CHUNKED) copy a row's scales 64 or 32 bytes at a
    // time, for SPC stages, into SBUFS buffers behind the ring (20 lines per stage; MXFP8 384 x 4096 x 4096 16.0 -> 13.5 us, on
    // 128 x 128 tiles up to a fifth less).  So does the narrow fp4 tile, whose stage takes 64 bytes (5 % less).  With fewer rows the
    // start counts more, which takes longer so (32 x 32 tile, fp8 5 x 4352 x 640 3.4 -> 3.6 us), and where a stage takes 16 bytes of
    // a row there is nothing to gain (fp4 on 96 x 64: 1 % more): these copy dwords into the stage itself.
    static constexpr int SPS = Op::SCALED ? SB / KB : 0;
    static constexpr bool CHUNKED = Op::SCALED && ((ROWS >= 160 && SPS <= 2) || SPS >= 16);
    static constexpr int STAGE_SPS = CHUNKED ? 0 : SPS;                        // (scale dwords inside a stage)
    static constexpr int SPIECES = ROWS * STAGE_SPS / 64, NSW = (SPIECES + NW - 1) / NW; // 64-dword scale pieces; per wave
    static constexpr int NV = NPW + NSW;                                  // copies a wave issues per stage
    static constexpr int STAGE = ROWS * SB + ROWS * STAGE_SPS * 4;
    // (the chunk of the stage that is being copied finds a buffer whose last reader is past)
    static constexpr int scale_buffers(int scb) { return !CHUNKED ? 0 : 1 + (R - 1 + scb / 4 / SPS - 1) / (scb / 4 / SPS); }
    static constexpr int SCB = !CHUNKED ? 64 : R * STAGE + scale_buffers(64) * ROWS * 64 <= 160 * 1024 ? 64 : 32;
    static constexpr int SPC = CHUNKED ? SCB / 4 / SPS : 1, SBUFS = scale_buffers(SCB);
    static constexpr int SCALE_BYTES = SBUFS * ROWS * SCB;
    static constexpr int KR = SB / 2, RB = BN * 2, CB = RB / 16;          // BND: k rows of a stage, bytes and chunks per row
    static constexpr int AHEAD = NPW <= 8 ? 3 : 2;                        // ANY: stages a copying wave holds in registers
    static constexpr int RED_PITCH = BN + 4;                              // elements
    static constexpr int RED_BYTES = WK * BM * RED_PITCH * 4;
    static constexpr int LDS_BYTES = (R * STAGE + SCALE_BYTES > RED_BYTES ? R * STAGE + SCALE_BYTES : RED_BYTES);
    static_assert(BM % (16 * WM) == 0 && BN % (16 * WN) == 0, "wave tiles are made of 16x16 blocks");
    static_assert(KW % KB == 0 && SB <= 1024 && 1024 % SB == 0, "a k-group's part of a stage is whole k-steps");
    static_assert(PIECES % NW == 0 && (BM * SB) % 1024 == 0, "every wave issues the same number of 1 KiB copies, each of one operand");
    static_assert(!BND || (!Op::SCALED && FR == 1 && (NB & (NB - 1)) == 0), "the row-major form is for the 16-bit types");
    static_assert(!SKEW || (PIPE && !BND && !ANY && !Op::SCALED && R >= 4), "two stages have to have landed where one is multiplied");
    static_assert(!ANY || (PIPE && !Op::SCALED), "the register copies are the copying waves' and know no scales");
    static_assert(!ANY || !BND || A_PIECES % NW == 0, "which copies are B's is known at compile time");
    static_assert((ROWS * STAGE_SPS) % 64 == 0, "scale pieces are whole");
    static_assert(PIPE == (LW > 0), "where some waves only copy, all read the scales' arguments: the pipelined form");
    static_assert(!CHUNKED || (SCB / 4 % SPS == 0 && (SBUFS - 1) * SPC >= R - 1 && BM * SCB % 1024 == 0 && BN * SCB % 1024 == 0 && ROWS <= CW * 64),
                  "a chunk of scales is whole stages; a 1 KiB copy of them is of one operand; a thread can hold a row's");
    static_assert(LDS_BYTES <= 160 * 1024 && R >= 2 && R * NV + (CHUNKED ? ROWS * SCB / 1024 / NW + 1 : 0) < 64, "LDS capacity; vmcnt is a 6-bit count");
};

// The copies of a row-major B (BND): what lane `lane` of copy q of copying wave lw brings.  A stage is KR k rows of BN columns, a chunk
// eight columns of a k row.
template <class Cfg>
struct RingRowCopies {
    // the stage's row, and the chunk of it
    __host__ __device__ static __forceinline__ int row(int lw, int q, int lane) { return ((lw + q * Cfg::NW - Cfg::A_PIECES) * 64 + lane) / Cfg::CB; }
    __host__ __device__ static __forceinline__ int chunk(int row, int lane) { return (lane % Cfg::CB) ^ (swizzle_row_major<Cfg::BN>(row) << 1); }
    // first byte fetched of a k row: of the chunk that N ends in, and of those past it, the 16 that end there
    __host__ __device__ static __forceinline__ int byte(int n, int n0, int chunk)
    {
        const int at = n0 * 2 + chunk * 16, last = n * 2 - 16;
        return at < last ? at : last;
    }
    // k row fetched for row r of the matrix: of eight rows that K ends in, and of those past them, the eight that end there, as in A's chunk of the
    // same k.  base: the row that a stage's offsets are counted from.
    __host__ __device__ static __forceinline__ int source(int k, int r) { return (r | 7) < k ? r : k - 8 + (r & 7); }
    __host__ __device__ static __forceinline__ int base(int stage) { return stage * Cfg::KR > 8 ? stage * Cfg::KR - 8 : 0; }
};

// position of a row's 16-byte chunk is chunk ^ ring_swizzle(row)
template <int SB>
__device__ __forceinline__ int ring_swizzle(int row)
{
    return SB == 128 ? swizzle_chunk(row, 0) : (row & 15);
}

// position of a row's 16-byte piece of scales is piece ^ ring_scale_swizzle(row): the byte reads of 16 rows hit different banks
template <int SCB>
__device__ __forceinline__ int ring_scale_swizzle(int row)
{
    return (row / (256 / SCB)) % (SCB / 16);
}

template <int N>
__device__ __forceinline__ void ring_wait_and_barrier()
{
    // own copies up to the stage have landed, own fragment reads of the previous stage have returned; then everybody's
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"(N) : "memory");
}

// the K tail: of the 16 bytes of a fragment chunk only `valid` belong to the row, the last ones (valid >= 16: all)
__device__ __forceinline__ uint4 ring_chunk_mask(int valid)
{
    uint32_t m[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int n = 16 - valid - 4 * i;  // low bytes of the dword to clear
        m[i] = n <= 0 ? 0xFFFFFFFFu : (n >= 4 ? 0u : 0xFFFFFFFFu << (8 * n));
    }
    return make_uint4(m[0], m[1], m[2], m[3]);
}
__device__ __forceinline__ uint4 ring_masked(uint4 v, uint4 m) { return make_uint4(v.x & m.x, v.y & m.y, v.z & m.z, v.w & m.w); }

// the chunk without its first `bytes` bytes, an even number below 16 (from 16 on: anything)
__device__ __forceinline__ uint4 ring_shift_down(uint4 v, uint32_t bytes)
{
    const uint64_t lo = (uint64_t)v.y << 32 | v.x, hi = (uint64_t)v.w << 32 | v.z;
    const uint32_t bits = (bytes & 6) * 8;
    uint64_t low = lo >> bits | hi << 1 << (63 - bits), high = hi >> bits;
    if (bytes & 8) {
        low = high;
        high = 0;
    }
    return make_uint4((uint32_t)low, (uint32_t)(low >> 32), (uint32_t)high, (uint32_t)(high >> 32));
}

// Consecutive columns of an output row that one thread drains: 16 bytes of 16- and 32-bit outputs, 4 of one-byte outputs and, where a thread
// would have more than four such pieces, 8 (int8 by a word: 256 x 128 tiles 0.91 to 0.97 of the time with 4, 128 x 128 0.93 to 0.97; on 128 x
// 64, four pieces, 1.02).
// Half or a quarter of that on the narrow tiles, which have fewer elements than that many times their threads: the pieces of a thread are
// added and stored one after the other while most threads have none.  bf16 24 x 4096 x 4096 on 32 x 16 tiles 7.48 -> 7.09 us, 64 x 8192 x
// 1024 on 64 x 32 6.0 -> 5.5.
template <int KIND, class Cfg>
constexpr int ring_columns()
{
    int ne = out_bytes<KIND> == 2 || (out_bytes<KIND> == 1 && Cfg::BM * Cfg::BN > 16 * Cfg::THREADS) ? 8 : 4;
    while (out_bytes<KIND> > 1 && ne > 2 && Cfg::BM * Cfg::BN < ne * Cfg::THREADS)
        ne /= 2;
    return ne;
}
template <int KIND, class Cfg>
constexpr int ring_cols = ring_columns<KIND, Cfg>();
// What depends on the column only.  A thread drains the same columns of several rows and fetches these once (fetched with
// every row they cost bf16 1237 x 4100 x 2056 with a bias row 8 us).
template <int KIND, int NE, class Elem>
struct RingColumns {
    Elem bias[NE];
    float scale[NE];
    uint64_t qw[NE];
    __device__ __forceinline__ void load(const TileGemmParams& p, int gj)
    {
        if (p.bias != nullptr) {
#pragma unroll
            for (int e = 0; e < NE; ++e)
                bias[e] = reinterpret_cast<const Elem*>(p.bias)[min(gj + e, p.n - 1)];
        }
#pragma unroll
        for (int e = 0; e < NE; ++e) {
            scale[e] = KIND == OUT_W8A8_BF16 ? p.col_scale[min(gj + e, p.n - 1)] : 1.0f;
            qw[e] = out_quant<KIND> ? p.qwords[p.q_per_column ? min(gj + e, p.n - 1) : 0] : 0;
        }
    }
};
template <int KIND, int NE, class Elem>
__device__ __forceinline__ void ring_store(const TileGemmParams& p, Elem (&v)[NE], const RingColumns<KIND, NE, Elem>& cols, float rs, int gi, int gj)
{
    const long o = (long)gi * p.ldc + gj;
    const int live = min(NE, p.n - gj);
    const bool raw = KIND == OUT_W8A8_BF16 && p.acc_out != nullptr;
    if (p.c_in != nullptr) {
#pragma unroll
        for (int e = 0; e < NE; ++e)
            v[e] += reinterpret_cast<const Elem*>(p.c_in)[o + (e < live ? e : 0)];
    }
    if (p.bias != nullptr) {
#pragma unroll
        for (int e = 0; e < NE; ++e)
            v[e] += cols.bias[e];
    }
    if (!out_quant<KIND> && (p.relu & 1)) {
#pragma unroll
        for (int e = 0; e < NE; ++e)
            v[e] = v[e] > 0 ? v[e] : 0;
    }
    if (raw) {
#pragma unroll
        for (int e = 0; e < NE; ++e)
            if (e < live)
                p.acc_out[o + e] = (int32_t)v[e];
    }
    uint32_t bits[NE];
#pragma unroll
    for (int e = 0; e < NE; ++e)
        bits[e] = tstore_bits<KIND>(v[e], rs, cols.scale[e], cols.qw[e], p.q_per_column != 0, p.relu, p.out_kind);
    if ((KIND == OUT_F32 || KIND == OUT_I32) && p.atomic_add) {
#pragma unroll
        for (int e = 0; e < NE; ++e)
            if (e < live) {
                if (KIND == OUT_F32)
                    atomicAdd(reinterpret_cast<float*>(p.c) + o + e, __builtin_bit_cast(float, bits[e]));
                else
                    atomicAdd(reinterpret_cast<int*>(p.c) + o + e, (int)bits[e]);
            }
        return;
    }
    uint8_t* dst = reinterpret_cast<uint8_t*>(p.c) + o * out_bytes<KIND>;
    if (live == NE) {
        // Vector stores go to any address.  Non-temporal: C is not read again here, and written back from the L2s it slows the
        // next launch (2048 x 4096 x 4096 to f32: 82 us with plain stores, 67 with these).
        if constexpr (out_bytes<KIND> == 1) {
            uint32_t w[NE / 4];
#pragma unroll
            for (int i = 0; i < NE / 4; ++i)
                w[i] = bits[4 * i] | (bits[4 * i + 1] << 8) | (bits[4 * i + 2] << 16) | (bits[4 * i + 3] << 24);
            __builtin_memcpy(dst, w, NE);
        } else {
            constexpr int WORDS = NE * out_bytes<KIND> / 4;
            uint32_t w[WORDS];
#pragma unroll
            for (int i = 0; i < WORDS; ++i)
                w[i] = out_bytes<KIND> == 2 ? bits[(2 * i) % NE] | (bits[(2 * i + 1) % NE] << 16) : bits[i % NE];
            typedef uint32_t nt1 __attribute__((aligned(1)));
            typedef uint32_t nt2 __attribute__((ext_vector_type(2), aligned(1)));
            typedef uint32_t nt4 __attribute__((ext_vector_type(4), aligned(1)));
            if constexpr (WORDS == 1)
                __builtin_nontemporal_store(w[0], reinterpret_cast<nt1*>(dst));
            else if constexpr (WORDS == 2)
                __builtin_nontemporal_store(nt2{w[0], w[1]}, reinterpret_cast<nt2*>(dst));
            else
                __builtin_nontemporal_store(nt4{w[0], w[1], w[2], w[3]}, reinterpret_cast<nt4*>(dst));
        }
    } else {
#pragma unroll
        for (int e = 0; e < NE - 1; ++e)
            if (e < live) {
                if (out_bytes<KIND> == 4)
                    reinterpret_cast<uint32_t*>(dst)[e] = bits[e];
                else if (out_bytes<KIND> == 2)
                    reinterpret_cast<uint16_t*>(dst)[e] = (uint16_t)bits[e];
                else
                    dst[e] = (uint8_t)bits[e];
            }
    }
}

// Has arguments in scalar registers from here on: they arrive in one wait, where the compiler's own loads, each in front of its first
// use, stand one after the other.
template <class T>
__device__ __forceinline__ void ring_argument(const T v)
{
    asm volatile("" : : "s"(v));
}
template <class... T>
__device__ __forceinline__ void ring_arguments(const T... v)
{
    (ring_argument(v), ...);
}

// The kernel's arguments as they lie in memory.  What is in front of `rest` are the fourteen scalar registers that the hardware fills
// before a wave starts (the units are compiled with kernel argument preloading): tile, addresses and first copies do not wait 0.3 to
// 0.4 us for the argument load.  `rest` is read through this, where it is needed: taken from the kernel's parameter it is loaded on
// entry, all of it, and the registers that it takes away are missed (MXFP8 384 x 4096 x 4096 11.3 us for 10.9).
struct RingArguments {
    const uint8_t *a, *b;
    uint32_t lda_bytes, ldb_bytes;
    int m, n, k_bytes, grid, tiles_m, per_group;
    uint32_t magic, shift;
    TileGemmParams rest;
};
// (in the kernel's order, each aligned by itself)
static_assert(offsetof(RingArguments, a) == 0 && offsetof(RingArguments, b) == 8 && offsetof(RingArguments, lda_bytes) == 16 && offsetof(RingArguments, ldb_bytes) == 20 &&
                  offsetof(RingArguments, m) == 24 && offsetof(RingArguments, n) == 28 && offsetof(RingArguments, k_bytes) == 32 && offsetof(RingArguments, grid) == 36 &&
                  offsetof(RingArguments, tiles_m) == 40 && offsetof(RingArguments, per_group) == 44 && offsetof(RingArguments, magic) == 48 &&
                  offsetof(RingArguments, shift) == 52 && offsetof(RingArguments, rest) == 56 && alignof(TileGemmParams) == 8,
              "the parameters' offsets");
template <class Cfg>
__global__ void __launch_bounds__(Cfg::THREADS) gemm_tile_ring_kernel(const uint8_t* a, const uint8_t* b, const uint32_t lda_bytes, const uint32_t ldb_bytes, const int m, const int n, const int k_bytes,
                                                                     const int grid, const int tiles_m, const int per_group, const uint32_t magic, const uint32_t shift, const TileGemmParams)
{
    using Op = typename Cfg::Op;
    using Acc = typename Op::Acc;
    using Elem = typename Op::Elem;
    constexpr int BM = Cfg::BM, BN = Cfg::BN, MB = Cfg::MB, NB = Cfg::NB, FR = Cfg::FR, SB = Cfg::SB, R = Cfg::R, NW = Cfg::NW;
    constexpr int NPW = Cfg::NPW, NSW = Cfg::NSW, NV = Cfg::NV, CPR = Cfg::CPR;
    constexpr bool CHUNKED = Cfg::CHUNKED;
    extern __shared__ __align__(16) uint8_t smem[];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const bool loads = Cfg::LW == 0 || wave >= Cfg::CW, computes = Cfg::LW == 0 || wave < Cfg::CW;
    const int lw = Cfg::LW == 0 ? wave : wave - Cfg::CW;  // number among the waves that copy
    const int wk = wave / (Cfg::WM * Cfg::WN), wmn = wave % (Cfg::WM * Cfg::WN), wm = wmn % Cfg::WM, wn = wmn / Cfg::WM;
    const int l16 = lane & 15, lg = lane >> 4;

    const TileGemmParams& rest = reinterpret_cast<const RingArguments*>((const void*)__builtin_amdgcn_kernarg_segment_ptr())->rest;
    TileGemmParams p;
    p.a = a;
    p.b = b;
    p.m = m;
    p.n = n;
    p.k_bytes = k_bytes;
    p.lda_bytes = lda_bytes;
    p.ldb_bytes = ldb_bytes;
    // Has the cache lines of `rest` fetched, so that the drain's loads find them; behind the first copies, where the wait costs nothing.
    auto touch_arguments = [&]() __attribute__((always_inline)) { ring_arguments(rest.c, rest.ldc, rest.q_per_column); };
    // for the drain, in one wait
    auto drain_arguments = [&]() __attribute__((always_inline)) {
        p.c = rest.c;
        p.c_in = rest.c_in;
        p.bias = rest.bias;
        p.acc_out = rest.acc_out;
        p.row_scale = rest.row_scale;
        p.col_scale = rest.col_scale;
        p.ldc = rest.ldc;
        p.relu = rest.relu;
        p.out_kind = rest.out_kind;
        p.qwords = rest.qwords;
        p.q_per_column = rest.q_per_column;
        p.atomic_add = rest.atomic_add;
        ring_arguments(p.c, p.c_in, p.bias, p.acc_out, p.row_scale, p.col_scale, p.ldc, p.relu, p.out_kind, p.qwords, p.q_per_column, p.atomic_add);
    };
    const RingTile tile = RingTiles{grid, tiles_m, per_group, {magic, shift}}.tile(blockIdx.x);
    const int m0 = tile.row * BM, n0 = tile.column * BN;

    // ---- TLOAD addressing: piece w + q * NW of a stage, lane -> (row, position) linear, fetching chunk position ^ swizzle
    const int nst = (p.k_bytes + SB - 1) / SB;
    const int ncopy = Cfg::SKEW ? (p.k_bytes + 7 * 16 + SB - 1) / SB : nst;  // stages copied
    const bool k_tail = p.k_bytes % SB != 0;
    const uint32_t lds0 = lds_address(smem);
    auto piece_row = [&](int q) { return (lw + q * NW) * Cfg::RPP + lane / CPR; };
    auto piece_chunk = [&](int q) { return (lane % CPR) ^ ring_swizzle<SB>(piece_row(q)); };
    auto row_offset = [&](int q) -> uint32_t {
        const int r = piece_row(q);
        return lw + q * NW < Cfg::A_PIECES ? (uint32_t)(min(m0 + r, p.m - 1) * p.lda_bytes) : (uint32_t)(min(n0 + r - BM, p.n - 1) * p.ldb_bytes);
    };
    using RowCopies = RingRowCopies<Cfg>;
    auto nd_row = [&](int q) { return RowCopies::row(lw, q, lane); };
    auto nd_chunk = [&](int q) { return RowCopies::chunk(nd_row(q), lane); };
    auto nd_col = [&](int q) -> uint32_t { return (uint32_t)RowCopies::byte(p.n, n0, nd_chunk(q)); };
    // SKEW: a stage of a row is whole 128-byte lines, so it starts `skew` chunks ahead of its own k.  Of the chunks of a stage's lines
    // that belong to this k stage and to the one before, each stands where its k has it: fragment reads find it at the same place
    // in either buffer, and their banks are those of rows that start on a line.
    auto skewed_chunk = [&](int q) -> int {
        if constexpr (!Cfg::SKEW)
            return piece_chunk(q);
        const int skew = ((uint32_t)(uintptr_t)(lw + q * NW < Cfg::A_PIECES ? p.a : p.b) + row_offset(q)) >> 4 & 7;
        return (piece_chunk(q) + skew) % CPR - skew;
    };
    constexpr int LINE = Cfg::SKEW ? 128 : 0;  // (added to the lanes' offsets, taken off the base: they stay positive)
    uint32_t goff[NPW];
#pragma unroll
    for (int q = 0; q < NPW; ++q)
        goff[q] = Cfg::BND && lw + q * NW >= Cfg::A_PIECES ? (uint32_t)(nd_row(q) * p.ldb_bytes) + nd_col(q) : row_offset(q) + skewed_chunk(q) * 16 + LINE;
    // Scales in the stage: dword e = row * STAGE_SPS + d; without scale arrays the copies fetch bytes of A that are not used.
    // (All that depends on the scales' arguments is worked out by scale_arguments(), which a copying wave calls behind its first copies.)
    bool has_scales = false, short_scales = false;
    int scale_last = 0, scale_shift = 0;
    const uint8_t* sc_row[NSW > 0 ? NSW : 1];
    int sc_d[NSW > 0 ? NSW : 1], sc_last = 0;  // last scale dword of a row
    auto scale_arguments = [&]() __attribute__((always_inline)) {
        if constexpr (Op::SCALED) {
            p.sa = rest.sa;
            p.sb = rest.sb;
            p.scale_ld = rest.scale_ld;
            ring_arguments(p.sa, p.sb, p.scale_ld);
            has_scales = p.sa != nullptr;
            sc_last = has_scales ? p.scale_ld / 4 - 1 : 0;
            short_scales = CHUNKED && has_scales && p.scale_ld < 16;
            scale_last = CHUNKED ? p.scale_ld / 16 * 4 : 0;
            scale_shift = CHUNKED ? (4 - p.scale_ld / 4 % 4) % 4 : 0;
            if constexpr (NSW > 0) {
#pragma unroll
                for (int q = 0; q < NSW; ++q) {
                    const int e = ((lw + q * NW) % Cfg::SPIECES) * 64 + lane, r = e / Cfg::STAGE_SPS;
                    sc_d[q] = e % Cfg::STAGE_SPS;
                    sc_row[q] = !has_scales ? p.a : r < BM ? p.sa + (long)min(m0 + r, p.m - 1) * p.scale_ld : p.sb + (long)min(n0 + r - BM, p.n - 1) * p.scale_ld;
                }
            }
        }
    };
    // Scales in chunks: without scale arrays nothing is copied and the buffers hold E8M0 127 (selected per fragment, the scales cost
    // a VALU instruction and a wait for each in front of the matrix instructions).  A row's
    // last 16 bytes are the 16 that END there, so where scale_ld is no multiple of 16 its last dwords lie scale_shift further on; a
    // row shorter than that (K < 512) goes through registers, of the waves that multiply where others copy: these have nothing else under
    // way, while in a copying wave the wait for the scales was one for all stages copied behind them (MXFP8 2048 x 4096 x 384 on 128 x
    // 128 tiles 14.8 -> 14.2 us, 384 x 4096 x 384 7.75 -> 7.5).  Out of line: in the way, K of 512 and more took 2 % longer.
    auto issue_scales = [&](int chunk) __attribute__((always_inline)) {
        if constexpr (CHUNKED) {
            constexpr int SCB = Cfg::SCB, LANES = SCB / 16, RPI = 64 / LANES, COPIES = Cfg::ROWS / RPI;  // lanes per row, rows per copy
            const uint32_t dst = lds0 + R * Cfg::STAGE + (chunk % Cfg::SBUFS) * (Cfg::ROWS * SCB);
#pragma unroll
            for (int q = 0; q < (COPIES + NW - 1) / NW; ++q) {
                const int c = lw + q * NW, r = c * RPI + lane / LANES;
                if (COPIES % NW != 0 && c >= COPIES)
                    break;
                const int byte = min(chunk * SCB + ((lane % LANES) ^ ring_scale_swizzle<SCB>(r)) * 16, p.scale_ld - 16);
                const bool is_a = c * RPI < BM;
                const int row = is_a ? min(m0 + r, p.m - 1) : min(n0 + r - BM, p.n - 1);
                lds_dma16_off(is_a ? p.sa : p.sb, (uint32_t)(row * p.scale_ld + byte), dst + c * 1024);
            }
        }
    };
    uint32_t held_scales[3];
    const int held_row = tid;  // (a wave that multiplies)
    auto hold_short_scales = [&]() __attribute__((always_inline)) {
        if constexpr (CHUNKED) {
            if (__builtin_expect(short_scales, 0) && held_row < Cfg::ROWS) {
                const uint8_t* row = held_row < BM ? p.sa + (long)min(m0 + held_row, p.m - 1) * p.scale_ld : p.sb + (long)min(n0 + held_row - BM, p.n - 1) * p.scale_ld;
#pragma unroll
                for (int d = 0; d < 3; ++d)
                    held_scales[d] = *reinterpret_cast<const uint32_t*>(row + min(4 * d, p.scale_ld - 4));
            }
        }
    };
    auto write_short_scales = [&]() __attribute__((always_inline)) {
        if constexpr (CHUNKED) {
            if (__builtin_expect(short_scales, 0) && held_row < Cfg::ROWS) {
                uint8_t* at = smem + R * Cfg::STAGE + held_row * Cfg::SCB + ring_scale_swizzle<Cfg::SCB>(held_row) * 16 + scale_shift * 4;
#pragma unroll
                for (int d = 0; d < 3; ++d)
                    if (4 * d < p.scale_ld)
                        *reinterpret_cast<uint32_t*>(at + 4 * d) = held_scales[d];
            }
        }
    };
    auto fill_scales = [&]() __attribute__((always_inline)) {
        if constexpr (CHUNKED) {
            if (__builtin_expect(!has_scales, 0))
                for (int o = tid * 16; o < Cfg::SCALE_BYTES; o += Cfg::CW * 64 * 16)
                    *reinterpret_cast<uint4*>(smem + R * Cfg::STAGE + o) = make_uint4(0x7F7F7F7Fu, 0x7F7F7F7Fu, 0x7F7F7F7Fu, 0x7F7F7F7Fu);
        }
    };
    auto issue_operands = [&](int st, int buf) __attribute__((always_inline)) {
        const uint32_t dst = __builtin_amdgcn_readfirstlane(lds0 + buf * Cfg::STAGE);
        const long kb = (long)st * SB, kb_b = Cfg::BND ? (long)st * Cfg::KR * p.ldb_bytes : kb;
        if (Cfg::SKEW ? st == 0 || (st + 1) * SB > p.k_bytes : k_tail && st == nst - 1) {
#pragma unroll
            for (int q = 0; q < NPW; ++q) {
                const int piece = lw + q * NW;
                if (Cfg::BND && piece >= Cfg::A_PIECES) {
                    const int base_row = RowCopies::base(st), src = RowCopies::source(p.k_bytes / 2, st * Cfg::KR + nd_row(q));
                    lds_dma16_off(p.b + (long)base_row * p.ldb_bytes, (uint32_t)((src - base_row) * p.ldb_bytes) + nd_col(q), dst + piece * 1024);
                    continue;
                }
                const int at = min(st * SB + skewed_chunk(q) * 16, p.k_bytes - 16);
                const uint32_t off = row_offset(q) + (uint32_t)(Cfg::SKEW ? max(at, 0) : at);
                lds_dma16_off(piece < Cfg::A_PIECES ? p.a : p.b, off, dst + piece * 1024);
            }
        } else {
#pragma unroll
            for (int q = 0; q < NPW; ++q) {
                const int piece = lw + q * NW;
                lds_dma16_off((piece < Cfg::A_PIECES ? p.a + kb : p.b + kb_b) - LINE, goff[q], dst + piece * 1024);
            }
        }
    };
    auto issue_stage_scales = [&](int st, int buf) __attribute__((always_inline)) {
        if constexpr (NSW > 0) {
            const uint32_t dst = __builtin_amdgcn_readfirstlane(lds0 + buf * Cfg::STAGE);
#pragma unroll
            for (int q = 0; q < NSW; ++q)
                lds_dma4(sc_row[q] + 4 * min(st * Cfg::STAGE_SPS + sc_d[q], sc_last), dst + Cfg::ROWS * SB + ((lw + q * NW) % Cfg::SPIECES) * 256);
        }
        if constexpr (CHUNKED) {
            if (has_scales && !short_scales && st % Cfg::SPC == 0)  // ahead of the next stage's copies, which stages are counted by
                issue_scales(st / Cfg::SPC);
        }
    };
    auto issue = [&](int st, int buf) __attribute__((always_inline)) {
        issue_operands(st, buf);
        issue_stage_scales(st, buf);
    };

    Acc acc[MB][NB];
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                acc[i][j][r] = 0;

    // ---- fragments: chunk c0 + lg of row l16 of a block, c0 a multiple of 4, sits at position c0 ^ (lg ^ swizzle(l16))
    const uint32_t lane_x = (uint32_t)((lg ^ ring_swizzle<SB>(l16)) ^ (wk * (Cfg::KW / 16))) << 4;
    const uint32_t fa_row = (wm * Cfg::WTM + l16) * SB, fb_row = (BM + wn * Cfg::WTN + l16) * SB;
    // Scale bytes.  In the stage: k-step s, row block i at {sa_at, sb_at} + 4 s + i * 16 * 4 STAGE_SPS of the stage.  In chunks: at
    // {a, b} of scale_rows(st) + 4 s + i * 16 * SCB; a chunk's dwords are 4 bytes apart but for the swizzle, which touches the bits of
    // a row's 16-byte pieces only, and a wave's k-steps lie in one piece.
    struct ScaleRows {
        uint32_t a, b;
    };
    constexpr int SCALE_ROW = CHUNKED ? Cfg::SCB : Cfg::STAGE_SPS * 4;
    const uint32_t scale_lane = (CHUNKED ? R * Cfg::STAGE + ((ring_scale_swizzle<Cfg::SCB>(l16) * 16) ^ (wk * Cfg::KSTEPS * 4)) : Cfg::ROWS * SB + wk * Cfg::KSTEPS * 4) + lg;
    const uint32_t sa_at = scale_lane + (wm * Cfg::WTM + l16) * SCALE_ROW, sb_at = scale_lane + (BM + wn * Cfg::WTN + l16) * SCALE_ROW;
    auto scale_rows = [&](uint32_t st) __attribute__((always_inline)) -> ScaleRows {
        if constexpr (!CHUNKED)
            return {0, 0};
        else {
            static_assert(Cfg::KSTEPS <= 4 && R * Cfg::STAGE % 64 == 0 && (Cfg::ROWS * Cfg::SCB) % 64 == 0, "a wave's k-steps of a stage lie in one 16-byte piece");
            const uint32_t in_chunk = (st * Cfg::SPS * 4) % Cfg::SCB;
            const uint32_t buf = (st / Cfg::SPC % Cfg::SBUFS) * (Cfg::ROWS * Cfg::SCB) + (st * Cfg::SPS + wk * Cfg::KSTEPS >= (uint32_t)scale_last ? scale_shift * 4 : 0);
            return {(sa_at ^ in_chunk) + buf, (sb_at ^ in_chunk) + buf};
        }
    };
    // BND: this lane's 8 bytes of a k-step's first block, k rows 8 lg .. + 3
    const int nd_l = lg * 8 + (l16 >> 2);
    const uint32_t nd_at = BM * SB + (wk * (Cfg::KW / 2) + nd_l) * Cfg::RB + ((wn * (Cfg::WTN / 16) ^ swizzle_row_major<BN>(nd_l)) << 5) + (l16 & 3) * 8;
    // Fragment registers.  PIPE: B's fragments and A's last row block have two sets, alternating per k-step; the other row
    // blocks of A are refilled in place right after their last matrix instruction, several of them before the next k-step
    // reads them.
    constexpr int SETS = Cfg::PIPE ? 2 : 1, NMMA = MB * NB;
    uint4 fa[SETS][MB][FR], fb[SETS][NB][FR];
    uint32_t xa[SETS][MB], xb[SETS][NB];
    auto aset = [](int set, int i) constexpr { return i == MB - 1 ? set : 0; };
    // SKEW: a chunk that is `skew` chunks or less from its stage's end came with the next one's lines.  Rows of a lane are 16 apart and
    // so have one skew.  {a, b}[s]: where the lane's chunk of k-step s is; next_a, next_b: behind the stage.
    struct Skewed {
        uint32_t a[Cfg::SKEW ? Cfg::KSTEPS : 1], b[Cfg::SKEW ? Cfg::KSTEPS : 1];
    };
    bool next_a[Cfg::SKEW ? Cfg::KSTEPS : 1], next_b[Cfg::SKEW ? Cfg::KSTEPS : 1];
    if constexpr (Cfg::SKEW) {
        static_assert(FR == 1, "a fragment is one chunk");
        const int skew_a = ((uint32_t)(uintptr_t)p.a + (uint32_t)((m0 + wm * Cfg::WTM + l16) * p.lda_bytes)) >> 4 & 7;
        const int skew_b = ((uint32_t)(uintptr_t)p.b + (uint32_t)((n0 + wn * Cfg::WTN + l16) * p.ldb_bytes)) >> 4 & 7;
#pragma unroll
        for (int s = 0; s < Cfg::KSTEPS; ++s) {
            next_a[s] = wk * (Cfg::KW / 16) + s * 4 + lg + skew_a >= CPR;
            next_b[s] = wk * (Cfg::KW / 16) + s * 4 + lg + skew_b >= CPR;
        }
    }
    auto skewed = [&](int b) __attribute__((always_inline)) -> Skewed {
        Skewed r{};
        if constexpr (Cfg::SKEW) {
            const uint32_t here = b * Cfg::STAGE, behind = (b + 1 == R ? 0 : b + 1) * Cfg::STAGE;
#pragma unroll
            for (int s = 0; s < Cfg::KSTEPS; ++s) {
                r.a[s] = fa_row + (lane_x ^ (s << 6)) + (next_a[s] ? behind : here);
                r.b[s] = fb_row + (lane_x ^ (s << 6)) + (next_b[s] ? behind : here);
            }
        }
        return r;
    };
    auto read_a = [&](int set, int i, int s, int b, const ScaleRows& sc, const Skewed& sk) __attribute__((always_inline)) {
        if constexpr (Cfg::SKEW) {
            fa[set][i][0] = *reinterpret_cast<const uint4*>(smem + sk.a[s] + i * (16 * SB));
            return;
        }
        const uint8_t* base = smem + b * Cfg::STAGE;
#pragma unroll
        for (int f = 0; f < FR; ++f)
            fa[set][i][f] = *reinterpret_cast<const uint4*>(base + fa_row + i * (16 * SB) + (lane_x ^ ((s * 4 * FR + 4 * f) << 4)));
        if constexpr (Op::SCALED)
            xa[set][i] = (CHUNKED ? smem + sc.a : base + sa_at)[s * 4 + i * (16 * SCALE_ROW)];
    };
    auto read_b = [&](int set, int j, int s, int b, const ScaleRows& sc, const Skewed& sk) __attribute__((always_inline)) {
        if constexpr (Cfg::SKEW) {
            fb[set][j][0] = *reinterpret_cast<const uint4*>(smem + sk.b[s] + j * (16 * SB));
            return;
        }
        const uint8_t* base = smem + b * Cfg::STAGE;
        if constexpr (Cfg::BND) {
            const uint8_t* at = base + (nd_at ^ (j << 5)) + s * 32 * Cfg::RB;
            fb[set][j][0] = read_transposed_16(at, at + 4 * Cfg::RB);
            return;
        }
#pragma unroll
        for (int f = 0; f < FR; ++f)
            fb[set][j][f] = *reinterpret_cast<const uint4*>(base + fb_row + j * (16 * SB) + (lane_x ^ ((s * 4 * FR + 4 * f) << 4)));
        if constexpr (Op::SCALED)
            xb[set][j] = (CHUNKED ? smem + sc.b : base + sb_at)[s * 4 + j * (16 * SCALE_ROW)];
    };
    auto read_all = [&](int set, int s, int b, const ScaleRows& sc, const Skewed& sk) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < NB; ++j)
            read_b(set, j, s, b, sc, sk);
#pragma unroll
        for (int i = 0; i < MB; ++i)
            read_a(aset(set, i), i, s, b, sc, sk);
    };
    auto mma = [&](int set, int i, int j) __attribute__((always_inline)) {
        const int as = aset(set, i);
        Op::mma(acc[i][j], fa[as][i], fb[set][j], Op::SCALED ? (CHUNKED || has_scales ? xa[as][i] : 127u) : 0u, Op::SCALED ? (CHUNKED || has_scales ? xb[set][j] : 127u) : 0u);
    };
    // k-step s of the last stage may reach past K: the first K byte of it, and its fragments masked
    auto tail_start = [&](int s) { return (nst - 1) * SB + wk * Cfg::KW + s * Cfg::KB; };
    auto mask_all = [&](int set, int s) __attribute__((always_inline)) {
#pragma unroll
        for (int f = 0; f < FR; ++f) {
            const uint4 mask = ring_chunk_mask(p.k_bytes - (tail_start(s) + (4 * f + lg) * 16));
#pragma unroll
            for (int i = 0; i < MB; ++i)
                fa[aset(set, i)][i][f] = ring_masked(fa[aset(set, i)][i][f], mask);
#pragma unroll
            for (int j = 0; j < NB; ++j)
                fb[set][j][f] = ring_masked(fb[set][j][f], mask);
        }
    };

    // ---- the K loop
    using std::integral_constant;
    // the copying side of a barrier: `behind` later stages may still be in flight
    auto loader_barrier = [&](int behind) __attribute__((always_inline)) {
        static_for<R>([&](auto ac) {
            constexpr int a = decltype(ac)::value;
            if (behind == a)
                ring_wait_and_barrier<a * NV>();
        });
    };
    if constexpr (!Cfg::PIPE) {
        // Barrier st: stage st has landed and no wave reads stage st - 1 any more, whose buffer is refilled.
        if (loads) {
            if constexpr (CHUNKED)
                scale_arguments();
            hold_short_scales();
            fill_scales();
            issue_operands(0, 0);
            if constexpr (!CHUNKED)
                scale_arguments();
            issue_stage_scales(0, 0);
#pragma unroll
            for (int s = 1; s < R - 1; ++s)
                if (s < nst)
                    issue(s, s);
            touch_arguments();
            write_short_scales();
        }
        int buf = 0;
        auto step = [&](int st) __attribute__((always_inline)) {
            if (!loads)
                ring_wait_and_barrier<63>();
            else {
                loader_barrier(min(R - 2, nst - 1 - st));
                if (st + R - 1 < nst)
                    issue(st + R - 1, buf == 0 ? R - 1 : buf - 1);
            }
        };
        for (int st = 0; st < nst - 1; ++st) {
            const ScaleRows rows = scale_rows(st);
            step(st);
            if (computes)
                static_for<Cfg::KSTEPS>([&](auto sc) {
                    read_all(0, decltype(sc)::value, buf, rows, Skewed{});
#pragma unroll
                    for (int i = 0; i < MB; ++i)
#pragma unroll
                        for (int j = 0; j < NB; ++j)
                            mma(0, i, j);
                });
            buf = buf + 1 == R ? 0 : buf + 1;
        }
        const ScaleRows rows = scale_rows(nst - 1);
        step(nst - 1);
        if (computes)
            static_for<Cfg::KSTEPS>([&](auto sc) {
                constexpr int s = decltype(sc)::value;
                read_all(0, s, buf, rows, Skewed{});
                if (tail_start(s) >= p.k_bytes)
                    return;
                if (k_tail)
                    mask_all(0, s);
#pragma unroll
                for (int i = 0; i < MB; ++i)
#pragma unroll
                    for (int j = 0; j < NB; ++j)
                        mma(0, i, j);
            });
    } else {
        // Barrier st stands in front of or in the last k-step of stage st: every wave holds that k-step's fragments, so the stage's
        // buffer is refilled with stage st + R, and stage st + 1 has landed, whose first fragments are read under that
        // k-step's matrix instructions.
        static_assert(Cfg::LW > 0, "the pipelined form has waves that only copy");
        if (Cfg::ANY && !computes) {
            // A stage's chunks are loaded AHEAD stages before they are written.  Neither is ever skipped -- past the last
            // stage both repeat it, into a buffer that nobody reads any more -- so that the count of loads in flight is known.
            constexpr int G = Cfg::AHEAD;
            uint32_t row[NPW], chunk[NPW];
            uint4 held[G][NPW];
#pragma unroll
            for (int q = 0; q < NPW; ++q) {
                const bool rows_of_k = Cfg::BND && q * NW >= Cfg::A_PIECES;
                row[q] = rows_of_k ? nd_col(q) : row_offset(q);
                chunk[q] = rows_of_k ? 0 : piece_chunk(q) * 16;
            }
            auto load = [&](auto gc, int st) __attribute__((always_inline)) {
                const int stage = min(st, nst - 1);
                const uint32_t k0 = stage * SB;
                const int base_row = RowCopies::base(stage);
#pragma unroll
                for (int q = 0; q < NPW; ++q) {
                    if (Cfg::BND && q * NW >= Cfg::A_PIECES) {
                        const int src = RowCopies::source(p.k_bytes / 2, stage * Cfg::KR + nd_row(q));
                        held[decltype(gc)::value][q] = load_unaligned16(p.b + (long)base_row * p.ldb_bytes + ((uint32_t)((src - base_row) * p.ldb_bytes) + row[q]));
                        continue;
                    }
                    const uint32_t off = row[q] + min(k0 + chunk[q], (uint32_t)(p.k_bytes - 16));
                    held[decltype(gc)::value][q] = load_unaligned16((lw + q * NW < Cfg::A_PIECES ? p.a : p.b) + off);
                }
            };
            // BND: the chunk of a row that N ends in came as the 16 bytes that end there
            const bool n_tail = Cfg::BND && n0 + BN > p.n && p.n % 8 != 0;
            auto store = [&](auto gc, int b) __attribute__((always_inline)) {
#pragma unroll
                for (int q = 0; q < NPW; ++q) {
                    uint4 v = held[decltype(gc)::value][q];
                    if (Cfg::BND && q * NW >= Cfg::A_PIECES && n_tail)
                        v = ring_shift_down(v, (uint32_t)(n0 * 2 + nd_chunk(q) * 16) - row[q]);
                    *reinterpret_cast<uint4*>(smem + b * Cfg::STAGE + (lw + q * NW) * 1024 + lane * 16) = v;
                }
            };
            static_for<G>([&](auto gc) { load(gc, decltype(gc)::value); });
            static_for<R>([&](auto sc) {
                constexpr int s = decltype(sc)::value;
                store(integral_constant<int, s % G>{}, s);
                load(integral_constant<int, s % G>{}, s + G);
            });
            ring_wait_and_barrier<63>();
            touch_arguments();
            int buf = 0, st = 0;
            auto step = [&](auto gc) __attribute__((always_inline)) {
                constexpr integral_constant<int, (R + decltype(gc)::value) % G> g{};
                ring_wait_and_barrier<63>();
                store(g, buf);
                load(g, st + R + G);
                buf = buf + 1 == R ? 0 : buf + 1;
                ++st;
            };
#pragma unroll 1
            while (st + G < nst)
                static_for<G>([&](auto gc) { step(gc); });
            static_for<G - 1>([&](auto gc) {
                if (st < nst - 1)
                    step(gc);
            });
        } else if (!computes) {
            // (SKEW: two stages, copies, up to a stage more of them)
            // The first barrier stands behind one stage more than the multiplying waves need, not behind the whole ring: to issue that takes 1.3
            // to 2 us on a cold start, long after the first stage has landed.  First product at 1.55 instead of 1.95 us (MXFP8 384 x 4096 x 4096
            // on 96 x 64 tiles, launch 12.2 -> 11.8 us), 0.9 instead of 1.45 (bf16 2048 x 2048 x 4096 on 128 x 128, 32.0 -> 31.3); behind just what
            // they need it is 0.1 us earlier and the launch no shorter.
            constexpr int AHEAD = Cfg::SKEW ? 2 : 1, EARLY = AHEAD + 1;
            static_assert(EARLY < R, "the ring holds more than the first barrier waits for");
            static_for<R>([&](auto sc) {
                constexpr int s = decltype(sc)::value;
                if constexpr (s == EARLY)
                    loader_barrier(max(0, min(EARLY - AHEAD, ncopy - AHEAD)));
                if constexpr (s == 0) {
                    issue_operands(0, 0);
                    scale_arguments();
                    issue_stage_scales(0, 0);
                } else if (s < ncopy) {
                    issue(s, s);
                }
            });
            touch_arguments();
            int buf = 0;
            for (int st = 0; st < nst - 1; ++st) {
                loader_barrier(max(0, min(R - 1 - AHEAD, ncopy - 1 - AHEAD - st)));
                if (st + R < ncopy)
                    issue(st + R, buf);
                buf = buf + 1 == R ? 0 : buf + 1;
            }
        } else {
            scale_arguments();
            touch_arguments();
            hold_short_scales();
            fill_scales();
            write_short_scales();
            // the scale addresses of a stage and the next one's: computed a stage ahead, off the way from barrier to matrix instruction
            ScaleRows rows = scale_rows(0), next_rows = scale_rows(1);
            Skewed skew = skewed(0), next_skew = skewed(1);
            ring_wait_and_barrier<63>();
            read_all(0, 0, 0, rows, skew);
            int buf = 0, st = 0;
            // One k-step on register set SET.  NEXT: under its matrix instructions the fragments of the next one are read, k-step rs of ring
            // buffer rb.  BARRIER: that one is another stage's.
            // The barrier waits for the wave's own reads, the last of which go out a row of matrix instructions before the k-step's end:
            // it stands a row into the last k-step, so that two rows cover them (and nothing is moved across it: the compiler put
            // all but one of that row's instructions behind it).  128 x 128 tiles 700 -> 680 clocks a stage, 256 x 128 1211 -> 1160, 192 x
            // 128 970 -> 953, MXFP8 on 96 x 64 936 -> 880.
            auto k_step = [&](auto setc, auto nextc, auto barrierc, int rs, int rb, const ScaleRows& rsc, const Skewed& rsk) __attribute__((always_inline)) {
                constexpr int SET = decltype(setc)::value;
                constexpr bool NEXT = decltype(nextc)::value, BARRIER = decltype(barrierc)::value;
                constexpr int BAR = BARRIER && MB > 1 && NMMA >= 6 ? NB : 0;
                static_for<NMMA>([&](auto xc) {
                    constexpr int x = decltype(xc)::value, i = x / NB, j = x % NB;
                    if constexpr (BARRIER && x == BAR) {
                        __builtin_amdgcn_sched_barrier(0);
                        ring_wait_and_barrier<63>();
                    }
                    mma(SET, i, j);
                    constexpr int y = x - BAR, AL = NB < NMMA - BAR ? NB : NMMA - BAR - 1;
                    if constexpr (NEXT && y >= 0 && (y < NB || y == AL || (j == NB - 1 && i < MB - 1))) {
                        __builtin_amdgcn_sched_barrier(0);
                        if constexpr (y < NB)
                            read_b(SET ^ 1, y, rs, rb, rsc, rsk);
                        if constexpr (y == 0)
                            static_for<BAR / NB>([&](auto rc) { read_a(0, decltype(rc)::value, rs, rb, rsc, rsk); });
                        if constexpr (y == AL)
                            read_a(SET ^ 1, MB - 1, rs, rb, rsc, rsk);
                        if constexpr (j == NB - 1 && i < MB - 1)
                            read_a(0, i, rs, rb, rsc, rsk);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                });
            };
            auto body = [&](auto parc) __attribute__((always_inline)) {
                constexpr int PAR = decltype(parc)::value;
                const int nbuf = buf + 1 == R ? 0 : buf + 1;
                static_for<Cfg::KSTEPS>([&](auto sc) {
                    constexpr int s = decltype(sc)::value;
                    constexpr integral_constant<int, (PAR + s) & 1> set{};
                    if constexpr (s + 1 < Cfg::KSTEPS)
                        k_step(set, std::true_type{}, std::false_type{}, s + 1, buf, rows, skew);
                    else
                        k_step(set, std::true_type{}, std::true_type{}, 0, nbuf, next_rows, next_skew);
                });
                buf = nbuf;
                ++st;
                rows = next_rows;
                next_rows = scale_rows(st + 1);
                skew = next_skew;
                next_skew = skewed(nbuf + 1 == R ? 0 : nbuf + 1);
            };
            // The last stage: nothing behind it, and K may end in it.  One piece of code for both kinds of K, of the steps that the loop has: next to
            // a copy for whole stages only and one that masks, read by read, the accumulators had registers of their own in either (128 x 128 tiles
            // 200 for 128, rows on any byte 238 for 162, on 96 x 64 tiles 256 for 156), and rows on any byte, whose K hardly ever is whole
            // stages, took longer: bf16 1 x 469 x 739 on 96 x 64 tiles 9.3 us before there were two, 9.6 with two, 8.95 now; 2198 x 3141 x 931 on
            // 128 x 64 58.3, 60.2, 57.3.  All stages through the loop, one more barrier and the reads in it for nothing: whole stages 1 % longer.
            auto last = [&](auto parc) __attribute__((always_inline)) {
                static_for<Cfg::KSTEPS>([&](auto sc) {
                    constexpr int s = decltype(sc)::value;
                    constexpr integral_constant<int, (decltype(parc)::value + s) & 1> set{};
                    if (tail_start(s) >= p.k_bytes)
                        return;
                    if (k_tail)  // (masks always: whole stages 2.5 % longer)
                        mask_all(set, s);
                    k_step(set, integral_constant<bool, (s + 1 < Cfg::KSTEPS)>{}, std::false_type{}, s + 1, buf, rows, skew);
                });
            };
            if constexpr (Cfg::KSTEPS % 2 == 0) {
                while (st < nst - 1)
                    body(integral_constant<int, 0>{});
                last(integral_constant<int, 0>{});
            } else {  // the register sets change places from stage to stage
                while (st + 2 < nst) {
                    body(integral_constant<int, 0>{});
                    body(integral_constant<int, 1>{});
                }
                if (st + 1 < nst) {
                    body(integral_constant<int, 0>{});
                    last(integral_constant<int, 1>{});
                } else {
                    last(integral_constant<int, 0>{});
                }
            }
        }
    }

    drain_arguments();
    // ---- TSTORE: the k-groups' partial sums meet in LDS (the ring is free), are added in group order and leave as up to 16
    // bytes per thread and row.  A block is transposed in its lanes: lane (l16, lg) holds row l16, columns 4 lg .. + 3.
    auto drain = [&](auto kc) __attribute__((always_inline)) {
        constexpr int KIND = decltype(kc)::value, NE = ring_cols<KIND, Cfg>, CT = BN / NE, RSTEP = Cfg::THREADS / CT;
        static_assert(Cfg::THREADS % CT == 0, "a thread keeps its columns from row to row");
        constexpr int VW = NE < 4 ? NE : 4;
        typedef Elem Piece __attribute__((ext_vector_type(VW)));
        const int c = (tid % CT) * NE, gj = n0 + c;
        // (what the columns and the first row bring is fetched while the sums are exchanged)
        RingColumns<KIND, NE, Elem> cols;
        cols.load(p, min(gj, p.n - 1));
        float rs = KIND == OUT_W8A8_BF16 ? p.row_scale[min(m0 + tid / CT, p.m - 1)] : 1.0f;
        __syncthreads();
        Elem* red = reinterpret_cast<Elem*>(smem) + wk * (BM * Cfg::RED_PITCH);
        if (computes) {
#pragma unroll
            for (int i = 0; i < MB; ++i)
#pragma unroll
                for (int j = 0; j < NB; ++j)
                    *reinterpret_cast<Acc*>(red + (wm * Cfg::WTM + i * 16 + l16) * Cfg::RED_PITCH + wn * Cfg::WTN + j * 16 + 4 * lg) = acc[i][j];
        }
        __syncthreads();
        if (gj >= p.n)
            return;
        auto drain_row = [&](int r) __attribute__((always_inline)) {
            Elem v[NE];
#pragma unroll
            for (int e = 0; e < NE; ++e)
                v[e] = 0;
#pragma unroll
            for (int g = 0; g < Cfg::WK; ++g)
#pragma unroll
                for (int q = 0; q < NE / VW; ++q) {
                    const Piece x = *reinterpret_cast<const Piece*>(reinterpret_cast<const Elem*>(smem) + (g * BM + r) * Cfg::RED_PITCH + c + VW * q);
#pragma unroll
                    for (int e = 0; e < VW; ++e)
                        v[VW * q + e] += x[e];
                }
            const float row_scale = rs;
            if (KIND == OUT_W8A8_BF16)
                rs = p.row_scale[min(m0 + r + RSTEP, p.m - 1)];
            ring_store<KIND>(p, v, cols, row_scale, m0 + r, gj);
        };
        // (Where a thread has more than one row piece, four of them in flight, eight of sixteen: one after the other each waits for its LDS
        // reads, which showed where four waves multiply and fewer threads drain.  256 x 128 tiles, bf16 1536 x 2560 x 640 14.5 -> 13.9 us, W8A8
        // 512 x 1024 x 1024 0.95 of before; with eight in flight int8 to int32 512 x 1024 x 1024 11.95 -> 11.7 us, but W8A8 on 192 x 128 3 % more.)
        if constexpr (RSTEP < BM) {
            constexpr int FLIGHT = BM / RSTEP >= 16 ? 8 : 4;
#pragma unroll FLIGHT
            for (int r = tid / CT; r < BM && m0 + r < p.m; r += RSTEP)
                drain_row(r);
        } else {
#pragma unroll 1
            for (int r = tid / CT; r < BM && m0 + r < p.m; r += RSTEP)
                drain_row(r);
        }
    };
    if (p.out_kind == OUT_Q8)
        drain(std::integral_constant<int, OUT_Q8>{});
    else if (p.out_kind >= OUT_QF16)
        drain(std::integral_constant<int, OUT_QF16>{});
    else if constexpr (std::is_same<Elem, int32_t>::value) {
        if (p.out_kind == OUT_I32)
            drain(std::integral_constant<int, OUT_I32>{});
        else
            drain(std::integral_constant<int, OUT_W8A8_BF16>{});
    } else {
        if (p.out_kind == OUT_F32)
            drain(std::integral_constant<int, OUT_F32>{});
        else if (p.out_kind == OUT_F16)
            drain(std::integral_constant<int, OUT_F16>{});
        else
            drain(std::integral_constant<int, OUT_BF16>{});
    }
}

}  // namespace ptoamd
