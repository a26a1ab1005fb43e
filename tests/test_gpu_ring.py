"""The deep-ring kernel's tile shapes at the sizes where they can go wrong: one row less and a few columns more than a tile,
one chunk of K, a stage and four bytes, fewer stages than the ring holds and more, against the CPU oracle."""
import numpy as np
import pytest
import torch

from oracle import binding as ob
from test_gpu_parity import (PA_T, _mx_inputs, _mx_unpack, _w8a8_reference, bf16_bits, bf16_to_f32, check_f32_drain, dev, host, pa,  # noqa: F401
                             relerr, tile_env)

pytestmark = pytest.mark.gpu

# rows, columns, bytes of K per stage (plain types, block-scaled types)
SHAPES = [(32, 16, 1024, 1024), (32, 32, 512, 512), (64, 32, 512, 512), (64, 64, 256, 256), (96, 64, 256, 256), (128, 64, 256, 256),
          (128, 128, 128, 128), (192, 128, 128, None), (256, 128, 128, None)]


def _sizes(shape, scaled):
    bm, bn, stage = SHAPES[shape][0], SHAPES[shape][1], SHAPES[shape][3 if scaled else 2]
    ks = (128, stage + 128, 6 * stage + 256) if scaled else (16, stage + 4, 2 * stage, 6 * stage + 36)
    return [(m, n, kb) for kb, (m, n) in zip(ks, ((bm - 1, bn + 3), (1, bn), (bm + 1, 2 * bn + 1), (bm, bn - 1)))]


@pytest.mark.parametrize("shape", range(9))
@pytest.mark.parametrize("kind", ["bf16", "f16", "i8"])
def test_plain_types(pa, oracle, kind, shape):  # noqa: F811
    r = np.random.default_rng(shape)
    for m, n, kb in _sizes(shape, False):
        k = kb if kind == "i8" else kb // 2
        if kind == "i8":
            a, b = (r.integers(-128, 128, (x, k)).astype(np.int8) for x in (m, n))
            da, db, ta, tc, ref = dev(a), dev(b), pa.I8, pa.I32, oracle.matmul_i8(a, b, b_dn=True)
        else:
            conv = (lambda x: x.astype(np.float16).view(np.uint16)) if kind == "f16" else bf16_bits
            a, b = (conv(r.uniform(-1, 1, (x, k)).astype(np.float32)) for x in (m, n))
            tdt = torch.float16 if kind == "f16" else torch.bfloat16
            da, db, ta, tc = dev(a).view(tdt), dev(b).view(tdt), pa.F16 if kind == "f16" else pa.BF16, pa.F32
            ref = (oracle.matmul_f16 if kind == "f16" else oracle.matmul_bf16)(a, b, b_dn=True)
        with tile_env(PTOAMD_RING=shape):
            got = host(pa.gemm(da, db, ta, tc, pa.B_DN))
            assert pa.last_kernel().startswith(f"tile{SHAPES[shape][0]}x{SHAPES[shape][1]}_dtl"), pa.last_kernel()
        if kind == "i8":
            assert np.array_equal(got, ref), (m, n, k)
        else:
            fa, fb = (x.view(np.float16).astype(np.float64) if kind == "f16" else bf16_to_f32(x).astype(np.float64) for x in (a, b))
            check_f32_drain(got, ref, np.abs(fa) @ np.abs(fb).T, k, f"{kind} {m}x{n}x{k} shape {shape}")


@pytest.mark.parametrize("shape", [1, 3, 4, 5, 6, 7, 8])
@pytest.mark.parametrize("kind", ["bf16", "f16", "i8"])
def test_rows_on_any_byte(pa, kind, shape):  # noqa: F811
    """Rows that start on any byte (16-bit types: on any element), from one chunk of K to more stages than ring and registers
    hold, the operands inside larger allocations whose other elements are NaN (int8: not zero): exact products of small
    whole numbers."""
    esz = 1 if kind == "i8" else 2
    tdt, t, tc = {"bf16": (torch.bfloat16, pa.BF16, pa.F32), "f16": (torch.float16, pa.F16, pa.F32), "i8": (torch.int8, pa.I8, pa.I32)}[kind]
    gen = torch.Generator(device="cuda").manual_seed(shape)
    bm, bn, stage = SHAPES[shape][:3]
    for m, n, kb in [(bm - 1, bn + 3, 18), (1, bn, stage + 6), (bm + 1, 2 * bn + 1, 2 * stage + 14), (bm, bn - 1, 4 * stage), (bm + 2, bn + 1, 9 * stage + 38)]:
        k = kb // esz + (1 if kb != 4 * stage else 0)

        def rows(count, pitch, start):  # whole numbers of -7 .. 7, all sums below 2^24
            flat = torch.full((start + count * pitch + 8,), 99 if kind == "i8" else float("nan"), device="cuda").to(tdt)
            view = flat[start:start + count * pitch].view(count, pitch)
            view[:, :k] = torch.randint(-7, 8, (count, k), generator=gen, device="cuda").to(tdt)
            return view
        for pitch in (k, k + 3):
            a, b = rows(m, pitch, 1), rows(n, pitch, 3)
            with tile_env(PTOAMD_RING=shape):
                got = pa.gemm(a, b, t, tc, pa.B_DN, k=k)
                assert pa.last_kernel() == f"tile{bm}x{bn}_any_{kind}", pa.last_kernel()
            assert torch.equal(got.double(), a[:, :k].double() @ b[:, :k].double().t()), (m, n, k, pitch)
    if kind == "i8":  # the W8A8 entry point takes the same kernels
        sa, sb = (torch.rand(x, generator=gen, device="cuda") for x in (m, n))
        with tile_env(PTOAMD_RING=shape):
            out = pa.gemm_w8a8(a[:, :k].contiguous(), b[:, :k].contiguous(), sa, sb)
            assert pa.last_kernel() == f"tile{bm}x{bn}_any_i8", pa.last_kernel()
        assert torch.equal(out, (got.float() * sa[:, None] * sb[None, :]).to(torch.bfloat16))


@pytest.mark.parametrize("shape", [1, 3, 4, 5, 6, 7, 8])
@pytest.mark.parametrize("kind", ["bf16", "f16"])
def test_row_major_b_rows_on_any_element(pa, kind, shape):  # noqa: F811
    """B as [K][N], no workspace, rows that start on any element and end anywhere in a chunk of eight columns (one chunk of columns, a tile
    and part of one, two tiles and one to seven columns), K from one chunk of eight rows to more stages than ring and registers hold,
    ending anywhere in a chunk: exact products of small whole numbers, NaN around the operands."""
    tdt, t = (torch.float16, pa.F16) if kind == "f16" else (torch.bfloat16, pa.BF16)
    gen = torch.Generator(device="cuda").manual_seed(shape)
    bm, bn, stage = SHAPES[shape][:3]
    kr = stage // 2

    def rows(count, length, pitch, start):  # whole numbers of -7 .. 7, all sums below 2^24; nothing behind the last row's values
        flat = torch.full((start + (count - 1) * pitch + length,), float("nan"), device="cuda").to(tdt)
        view = flat.as_strided((count, length), (pitch, 1), start)
        view.copy_(torch.randint(-7, 8, (count, length), generator=gen, device="cuda"))
        return view
    for m, n, k in [(bm - 1, 9, 8), (1, bn - 1, 9), (bm, 8, kr + 3), (bm + 1, 2 * bn + 1, 2 * kr + 7), (bm, bn + 2, 4 * kr), (2, bn + 3, 4 * kr + 1), (bm - 1, 2 * bn + 4, 7 * kr + 2),
                    (3, bn + 5, 7 * kr - 4), (bm + 2, bn + 6, 9 * kr + 13), (bm, 2 * bn + 7, 9 * kr + 6)]:
        for wide, start in ((0, 0), (3, 1)):
            a, b = rows(m, k, k + wide, start), rows(k, n, n + wide, start)
            with tile_env(PTOAMD_RING=shape):
                got = pa.gemm(a, b, t, pa.F32, pa.B_ND)
                name = pa.last_kernel()
            in_place = n % 8 == 0 and k % 2 == 0 and wide == 0
            assert in_place or name == f"tile{bm}x{bn}_bnd_any_{kind}", (name, m, n, k)
            assert torch.equal(got.double(), a.double() @ b.double()), (m, n, k, wide)


def test_row_major_b_without_workspace_takes_the_form_for_any_row(pa):  # noqa: F811
    for m, n, k in [(18, 308, 7274), (2, 1020, 4474), (55, 287, 3027), (300, 2049, 1025)]:
        gen = torch.Generator(device="cuda").manual_seed(m)
        a, b = (torch.randint(-7, 8, x, generator=gen, device="cuda").to(torch.bfloat16) for x in ((m, k), (k, n)))
        got = pa.gemm(a, b, pa.BF16, pa.F32, pa.B_ND)
        assert "_bnd_any_" in pa.last_kernel(), pa.last_kernel()
        assert torch.equal(got.double(), a.double() @ b.double())


@pytest.mark.parametrize("shape", [3, 4, 6, 7])
@pytest.mark.parametrize("kind", ["bf16", "f16", "i8"])
def test_rows_on_16_bytes_off_the_lines(pa, kind, shape):  # noqa: F811
    """Rows that start on 16 bytes but not on 128: pitches that leave one, four and eight different offsets, A and B apart, K from the
    six stages on that whole lines are copied for (and a chunk less), ending on a stage, a chunk and inside one; what is around the operands is NaN (int8: not zero).
    The bits of the product of the same operands on whole lines."""
    esz = 1 if kind == "i8" else 2
    tdt, t, tc = {"bf16": (torch.bfloat16, pa.BF16, pa.F32), "f16": (torch.float16, pa.F16, pa.F32), "i8": (torch.int8, pa.I8, pa.I32)}[kind]
    gen = torch.Generator(device="cuda").manual_seed(shape)
    bm, bn, stage = SHAPES[shape][:3]

    def rows(values, pitch, start):  # (in bytes)
        flat = torch.full((start // esz + values.shape[0] * pitch // esz,), 99 if kind == "i8" else float("nan"), device="cuda").to(tdt)
        view = flat[start // esz:].view(values.shape[0], pitch // esz)[:, :values.shape[1]]
        view.copy_(values)
        return view
    for m, n, kb in [(bm - 1, bn + 3, 6 * stage - 16), (1, bn, 6 * stage), (bm + 1, 2 * bn + 1, 6 * stage + 20), (bm, bn - 1, 8 * stage - 112), (bm + 2, bn + 1, 9 * stage + 100)]:
        a, b = ((torch.rand((x, kb // esz), generator=gen, device="cuda") * 200 - 100).to(tdt) for x in (m, n))
        line = (kb + 127) // 128 * 128
        with tile_env(PTOAMD_RING=shape):
            ref = pa.gemm(rows(a, line, 0), rows(b, line, 0), t, tc, pa.B_DN)
            for pa_, sa, pb, sb in [(line + 16, 0, line + 16, 0), (line + 64, 32, line + 32, 112), (line, 48, line + 240, 0), (line + 128, 0, line, 96)]:
                got = pa.gemm(rows(a, pa_, sa), rows(b, pb, sb), t, tc, pa.B_DN)
                assert torch.equal(got, ref), (m, n, kb, pa_, sa, pb, sb)
        assert torch.isfinite(got.double()).all()


@pytest.mark.parametrize("shape", range(9))
@pytest.mark.parametrize("kind", ["bf16", "f16", "i8"])
def test_which_rows_are_copied_by_lines(pa, kind, shape):  # noqa: F811
    """The form for rows off the lines runs on the shapes with four stages in the ring from six stages of K on, and on no other: by the
    kernel's name, and exact products of small whole numbers either way."""
    esz = 1 if kind == "i8" else 2
    tdt, t, tc = {"bf16": (torch.bfloat16, pa.BF16, pa.F32), "f16": (torch.float16, pa.F16, pa.F32), "i8": (torch.int8, pa.I8, pa.I32)}[kind]
    gen = torch.Generator(device="cuda").manual_seed(shape)
    bm, bn, stage = SHAPES[shape][:3]
    for kb, pitch, start, off in [(6 * stage, 6 * stage + 16, 0, True), (6 * stage - 16, 6 * stage + 16, 0, False), (6 * stage, 6 * stage + 128, 0, False),
                                  (6 * stage, 6 * stage + 128, 64, True), (6 * stage + 36, 6 * stage + 68, 0, False), (7 * stage + 36, 7 * stage + 48, 80, True)]:
        def rows(count):  # whole numbers of -7 .. 7, all sums below 2^24
            flat = torch.full(((start + count * pitch) // esz,), 99 if kind == "i8" else float("nan"), device="cuda").to(tdt)
            view = flat[start // esz:].view(count, pitch // esz)[:, :kb // esz]
            view.copy_(torch.randint(-7, 8, view.shape, generator=gen, device="cuda"))
            return view
        a, b = rows(bm + 1), rows(2 * bn - 1)
        with tile_env(PTOAMD_RING=shape):
            got = pa.gemm(a, b, t, tc, pa.B_DN)
            name = pa.last_kernel()
        form = "dtl_lines" if off and shape in (3, 4, 6, 7) else "dtl"
        assert name == f"tile{bm}x{bn}_{form}_{kind}", (kb, pitch, start, name)
        assert torch.equal(got.double(), a.double() @ b.double().t()), (kb, pitch, start)


def test_rows_copied_by_lines_beyond_2_gib(pa):  # noqa: F811
    """Lane offsets past 2^31 bytes: rows 17 MB apart."""
    m, n, k, pitch = 130, 65, 1024, (17 << 20) // 2 + 8
    gen = torch.Generator(device="cuda").manual_seed(0)
    a = torch.empty(m * pitch, dtype=torch.bfloat16, device="cuda").view(m, pitch)[:, :k]
    a.copy_(torch.randint(-7, 8, (m, k), generator=gen, device="cuda"))
    b = torch.randint(-7, 8, (n, k), generator=gen, device="cuda").to(torch.bfloat16)
    with tile_env(PTOAMD_RING=3):
        got = pa.gemm(a, b, pa.BF16, pa.F32, pa.B_DN)
        assert pa.last_kernel() == "tile64x64_dtl_lines_bf16", pa.last_kernel()
    assert torch.equal(got.double(), a.double() @ b.double().t())


@pytest.mark.parametrize("shape", range(9))
@pytest.mark.parametrize("kind", ["bf16", "f16"])
def test_row_major_b(pa, oracle, kind, shape):  # noqa: F811
    """B as [K][N] with columns that end in part of a tile and rows at a wider pitch (the columns past N hold NaN), K ending
    inside a stage and inside a chunk of eight rows: bit for bit the product with the same B given column-major."""
    r = np.random.default_rng(100 + shape)
    tdt, t = (torch.float16, pa.F16) if kind == "f16" else (torch.bfloat16, pa.BF16)
    for m, n, kb in _sizes(shape, False):
        n, k = (n + 7) // 8 * 8, kb // 2
        a, b = (torch.from_numpy(r.uniform(-1, 1, x).astype(np.float32)).to(tdt).cuda() for x in ((m, k), (k, n)))
        wide = torch.full((k, n + 10), float("nan"), dtype=tdt, device="cuda")
        wide[:, :n] = b
        with tile_env(PTOAMD_RING=shape):
            same = pa.gemm(a, b.t().contiguous(), t, pa.F32, pa.B_DN)
            got = pa.gemm(a, b, t, pa.F32, pa.B_ND)
            pitched = pa.gemm(a, wide, t, pa.F32, pa.B_ND, n=n)
            assert pa.last_kernel() == f"tile{SHAPES[shape][0]}x{SHAPES[shape][1]}_bnd_{kind}", pa.last_kernel()
        assert torch.equal(got, same) and torch.equal(pitched, same), (m, n, k)
        ref = a.double() @ b.double()  # (f32 sums of k products, each of them exact)
        bound = k * 2.0 ** -23 * (a.double().abs() @ b.double().abs()) + 1e-30
        assert bool(((got.double() - ref).abs() <= bound).all()), (m, n, k)


@pytest.mark.parametrize("k", [64, 128, 320])
@pytest.mark.parametrize("kind", ["bf16", "f16"])
def test_row_major_b_256x256(pa, kind, k):  # noqa: F811
    """The 256 x 256 tile's row-major form over one, two and five slabs, with a last row of tiles that is not full and tail
    columns that run on the deep-ring kernel: bits of the column-major product where that runs on the same tile."""
    m, n = 4090, 4112
    gen = torch.Generator(device="cuda").manual_seed(k)
    tdt, t = (torch.float16, pa.F16) if kind == "f16" else (torch.bfloat16, pa.BF16)
    a, b = (torch.rand(x, generator=gen, device="cuda").sub(0.5).to(tdt) for x in ((m, k), (k, n)))
    got = pa.gemm(a, b, t, pa.F32, pa.B_ND)
    assert pa.last_kernel() == f"tile256x256w8_bnd_{kind}", pa.last_kernel()
    same = pa.gemm(a, b.t().contiguous(), t, pa.F32, pa.B_DN)
    assert torch.equal(got[:, :4096], same[:, :4096])
    ref, mag = a.double() @ b.double(), a.double().abs() @ b.double().abs()
    assert bool(((got.double() - ref).abs() <= k * 2.0 ** -23 * mag).all())


@pytest.mark.parametrize("shape", range(7))
@pytest.mark.parametrize("ta,tb", [(ob.E4M3, ob.E4M3), (ob.E5M2, ob.E4M3), (ob.E4M3, ob.E5M2), (ob.E5M2, ob.E5M2), (ob.E2M1, ob.E2M1)])
def test_block_scaled_types(pa, oracle, ta, tb, shape):  # noqa: F811
    r = np.random.default_rng(shape + 16 * ta + tb)
    fp4 = ta == ob.E2M1
    for m, n, kb in _sizes(shape, True):
        k = 2 * kb if fp4 else kb
        a, _, sa, sb = _mx_inputs(r, ta, m, n, k)
        _, b, _, _ = _mx_inputs(r, tb, m, n, k)
        ref = oracle.matmul_mx(a, b, sa, sb, m, k, n, ta, tb)
        with tile_env(PTOAMD_RING=shape):
            got = host(pa.gemm_mx(dev(a), dev(b), dev(sa), dev(sb), m, n, k, PA_T[ta], PA_T[tb], pa.F32))
            assert pa.last_kernel().startswith(f"tile{SHAPES[shape][0]}x{SHAPES[shape][1]}_dtl"), pa.last_kernel()
        ua = _mx_unpack(oracle, a, ta) * np.repeat(2.0 ** (sa.astype(np.float64) - 127), 32, 1)
        ub = _mx_unpack(oracle, b, tb) * np.repeat(2.0 ** (sb.astype(np.float64) - 127), 32, 1)
        # (the fp8 form of the scaled instruction keeps about 13 bits below the largest of a block's products: 2^-11 of sum|a||b|)
        check_f32_drain(got, ref, np.abs(ua) @ np.abs(ub).T, k, f"MX {ta}x{tb} {m}x{n}x{k} shape {shape}",
                        max_rel=1e-4 if fp4 else 1e-3, eps=None if fp4 else 2.0 ** -11)


@pytest.mark.parametrize("shape", range(7))
@pytest.mark.parametrize("fp4", [False, True])
def test_block_scales_over_several_chunks(pa, oracle, fp4, shape):  # noqa: F811
    """Scales are copied 1024 or 2048 elements of K at a time: K of several such chunks, the last one short, its rows' scales
    ending on 16 bytes and off them; and rows of scales shorter than 16 bytes."""
    r = np.random.default_rng(400 + shape)
    bm, bn = SHAPES[shape][:2]
    t = ob.E2M1 if fp4 else ob.E4M3
    for m, n, k in ((bm + 1, bn - 1, 2560), (bm - 1, bn + 3, 6400 if fp4 else 6272), (bm, bn + 1, 256), (1, bn + 1, 256 if fp4 else 384)):
        one = 2 if fp4 else 0x38  # 1.0; the sign bit of a random half of the codes
        a, b = ((one | (r.integers(0, 2, (x, k)) << (3 if fp4 else 7))).astype(np.uint8) for x in (m, n))
        if fp4:
            a, b = ((x[:, 0::2] | (x[:, 1::2] << 4)).astype(np.uint8) for x in (a, b))
        sa, sb = (r.integers(120, 135, (x, k // 32)).astype(np.uint8) for x in (m, n))
        with tile_env(PTOAMD_RING=shape):
            got = host(pa.gemm_mx(dev(a), dev(b), dev(sa), dev(sb), m, n, k, PA_T[t], PA_T[t], pa.F32))
            assert pa.last_kernel().startswith(f"tile{bm}x{bn}_dtl"), pa.last_kernel()
        ua, ub = (_mx_unpack(oracle, x, t) * np.repeat(2.0 ** (s.astype(np.float64) - 127), 32, 1) for x, s in ((a, sa), (b, sb)))
        # (bounds as in test_block_scaled_types)
        check_f32_drain(got, ua @ ub.T, np.abs(ua) @ np.abs(ub).T, k, f"{m}x{n}x{k} shape {shape} fp4 {fp4}",
                        max_rel=1e-4 if fp4 else 1e-3, eps=None if fp4 else 2.0 ** -11)


@pytest.mark.parametrize("tile", [4, 5, 7])
@pytest.mark.parametrize("k", [512, 1536, 2560])
def test_block_scales_of_the_two_and_three_slab_tiles(pa, oracle, tile, k):  # noqa: F811
    """fp8 scales are copied 1024 elements of K at a time where they fit: half a chunk, one and a half, two and a half."""
    r = np.random.default_rng(tile + k)
    m, n = 259, 261
    a, b, sa, sb = _mx_inputs(r, ob.E4M3, m, n, k)
    with tile_env(PTOAMD_TILE=tile):
        got = host(pa.gemm_mx(dev(a), dev(b), dev(sa), dev(sb), m, n, k, pa.E4M3, pa.E4M3, pa.F32))
        assert "_dtl_fp8" in pa.last_kernel(), pa.last_kernel()
    ua, ub = (_mx_unpack(oracle, x, ob.E4M3) * np.repeat(2.0 ** (s.astype(np.float64) - 127), 32, 1) for x, s in ((a, sa), (b, sb)))
    check_f32_drain(got, ua @ ub.T, np.abs(ua) @ np.abs(ub).T, k, f"{m}x{n}x{k} tile {tile}", max_rel=1e-3, eps=2.0 ** -11)


def _fp8_operands(r, ta, tb, m, n, k):
    """Codes without NaN and infinities, on the device with rows at a wider pitch whose other bytes are NaN codes."""
    a, _, _, _ = _mx_inputs(r, ta, m, n, k)
    _, b, _, _ = _mx_inputs(r, tb, m, n, k)
    wide = []
    for x, pad in ((a, 4), (b, 20)):
        w = torch.full((x.shape[0], k + pad), 0x7F, dtype=torch.uint8, device="cuda")
        w[:, :k] = dev(x)
        wide.append(w[:, :k])
    return a, b, wide[0], wide[1]


@pytest.mark.parametrize("shape", range(7))
@pytest.mark.parametrize("ta,tb", [(ob.E4M3, ob.E4M3), (ob.E5M2, ob.E4M3), (ob.E4M3, ob.E5M2), (ob.E5M2, ob.E5M2)])
def test_fp8_without_scales(pa, oracle, ta, tb, shape):  # noqa: F811
    """No scale arrays, and a K that ends inside a stage, inside a fragment of 32 bytes and inside a chunk of 16."""
    r = np.random.default_rng(300 + shape + 16 * ta + tb)
    bm, bn, stage = SHAPES[shape][0], SHAPES[shape][1], SHAPES[shape][3]
    for m, n, k in ((bm - 1, bn + 3, 16), (1, bn, stage + 4), (bm + 1, 2 * bn + 1, 2 * stage), (bm, bn - 1, 6 * stage + 36)):
        a, b, da, db = _fp8_operands(r, ta, tb, m, n, k)
        ref = oracle.matmul_fp8(a, b, b_dn=True, a_type=ta, b_type=tb)
        with tile_env(PTOAMD_RING=shape):
            got = host(pa.gemm_fp8(da, db, PA_T[ta], PA_T[tb]))
            assert pa.last_kernel().startswith(f"tile{bm}x{bn}_dtl_fp8"), pa.last_kernel()
        mag = np.abs(_mx_unpack(oracle, a, ta)) @ np.abs(_mx_unpack(oracle, b, tb)).T
        # (the fp8 form of the scaled instruction keeps about 13 bits below the largest of a block's products: 2^-11 of sum|a||b|)
        check_f32_drain(got, ref, mag, k, f"fp8 {ta}x{tb} {m}x{n}x{k} shape {shape}", max_rel=1e-3, eps=2.0 ** -11)


@pytest.mark.parametrize("m,n,k,kernel", [(24, 1000, 1024, "tile32x16_dtl"), (384, 2048, 1060, "tile64x64_dtl"), (1000, 2048, 1024, "tile128x64_dtl"),
                                          (2048, 2560, 512, "tile128x128_dtl"), (1024, 6144, 1024, "tile256x128r3_dtl"), (4096, 4096, 256, "tile256x256w8_dtl")])
def test_fp8_without_scales_on_the_kernel_of_its_size(pa, m, n, k, kernel):  # noqa: F811
    """No switch set: products of small whole numbers, whose sums are exact, on the kernel that the sizes ask for."""
    gen = torch.Generator(device="cuda").manual_seed(k)
    a, b = (torch.randint(-2, 3, (x, k), generator=gen, device="cuda").float().to(torch.float8_e4m3fn).view(torch.uint8) for x in (m, n))
    got = pa.gemm(a, b, pa.E4M3, pa.F32, pa.B_DN)
    assert pa.last_kernel() == f"{kernel}_fp8_e4m3_e4m3", pa.last_kernel()
    value = lambda x: x.view(torch.float8_e4m3fn).double()  # noqa: E731
    assert torch.equal(got.double(), value(a) @ value(b).t())


@pytest.mark.parametrize("shape", [0, 3, 7])
def test_store_forms(pa, oracle, shape):  # noqa: F811
    """Accumulator input, bias, relu, 16-bit rows at an odd pitch, W8A8 with raw accumulators, per-column requantisation and
    atomic adds: integer and rounding steps are the oracle's, bit for bit."""
    r = np.random.default_rng(50 + shape)
    m, n, k = SHAPES[shape][0] + 5, SHAPES[shape][1] + 13, 324
    a, b = (r.integers(-128, 128, (x, k)).astype(np.int8) for x in (m, n))
    cin, bias = r.integers(-2 ** 30, 2 ** 30, (m, n)).astype(np.int32), r.integers(-1000, 1000, n).astype(np.int32)
    acc = oracle.matmul_i8(a, b, b_dn=True)
    sa, sb = r.uniform(0.001, 0.02, m).astype(np.float32), r.uniform(0.001, 0.02, n).astype(np.float32)
    words = np.array([(int(np.float32(r.uniform(1e-4, 1e-3)).view(np.uint32)) & 0xFFFFE000) | (int(r.integers(0, 16)) << 37) | (1 << 46)
                      for _ in range(n)], np.uint64)
    x, y = bf16_bits(r.uniform(-1, 1, (m, k)).astype(np.float32)), bf16_bits(r.uniform(-1, 1, (n, k)).astype(np.float32))
    with tile_env(PTOAMD_RING=shape):
        got = host(pa.gemm(dev(a), dev(b), pa.I8, pa.I32, pa.B_DN, c_in=dev(cin), bias=dev(bias), relu=True))
        out, raw = pa.gemm_w8a8(dev(a), dev(b), dev(sa), dev(sb), want_acc=True)
        q8 = host(pa.gemm_requant(dev(a), dev(b), pa.I8, pa.I8, dev(words.view(np.int64)), per_column=True))
        summed = dev(cin)
        pa.gemm_atomic_add(summed, dev(a), dev(b), pa.I8)
        wide = torch.full((m, n + 3), 7.0, dtype=torch.bfloat16, device="cuda:0")
        dx, dy = dev(x).view(torch.bfloat16), dev(y).view(torch.bfloat16)
        f32 = host(pa.gemm(dx, dy, pa.BF16, pa.F32, pa.B_DN))
        pa.gemm(dx, dy, pa.BF16, pa.BF16, pa.B_DN, out=wide[:, :n])
        assert "_dtl_" in pa.last_kernel()
    assert np.array_equal(got, np.maximum((acc.astype(np.int64) + cin + bias).astype(np.int32), 0))
    ref_acc, ref_out = _w8a8_reference(oracle, a, b, sa, sb)
    assert np.array_equal(host(raw), ref_acc) and np.array_equal(host(out), ref_out)
    assert np.array_equal(q8.view(np.uint8).ravel(), np.asarray(oracle.store_quant(acc, ob.ST_I8, words, True)).view(np.uint8).ravel())
    assert np.array_equal(host(summed), (acc.astype(np.int64) + cin).astype(np.int32))
    assert np.array_equal(host(wide)[:, :n], oracle.store_f32(f32, ob.ST_BF16))
    assert bool((wide[:, n:] == 7.0).all())


@pytest.mark.parametrize("shape", [3, 5, 6, 7, 8])
@pytest.mark.parametrize("per_column", [False, True])
def test_one_byte_results_in_pieces(pa, oracle, per_column, shape):  # noqa: F811
    """A thread stores 4 or (shapes 6 to 8) 8 one-byte columns at a time: N ending on each of 8 columns of a piece, on rows at an odd
    pitch whose other columns are kept."""
    r = np.random.default_rng(60 + shape)
    m, k = SHAPES[shape][0] + 5, 196
    n_most = SHAPES[shape][1] + 16
    a, b = (r.integers(-128, 128, (x, k)).astype(np.int8) for x in (m, n_most))
    words = np.array([(int(np.float32(r.uniform(1e-4, 1e-3)).view(np.uint32)) & 0xFFFFE000) | (int(r.integers(0, 16)) << 37) | (1 << 46)
                      for _ in range(n_most if per_column else 1)], np.uint64)
    acc = oracle.matmul_i8(a, b, b_dn=True)
    for n in range(n_most - 8, n_most):
        w = words[:n] if per_column else words
        wide = torch.full((m, n + 6 + n % 2), 7, dtype=torch.int8, device="cuda")
        with tile_env(PTOAMD_RING=shape):
            pa.gemm_requant(dev(a), dev(b[:n].copy()), pa.I8, pa.I8, dev(w.view(np.int64)), per_column=per_column, out=wide[:, 3:3 + n])
            assert "_dtl_" in pa.last_kernel()
        ref = np.asarray(oracle.store_quant(acc[:, :n].copy(), ob.ST_I8, w, per_column)).view(np.int8).reshape(m, n)
        assert np.array_equal(host(wide)[:, 3:3 + n].view(np.int8), ref), n
        assert bool((wide[:, :3] == 7).all()) and bool((wide[:, 3 + n:] == 7).all()), n


@pytest.mark.parametrize("drain,m,n,k", [("column words", 3967, 2560, 320), ("column words", 1324, 6144, 168), ("raw", 3788, 3968, 384), ("atomic", 1981, 7296, 128)])
def test_drains_keep_off_the_two_slab_128x128_tile(pa, drain, m, n, k):  # noqa: F811
    """Drains that the 128 x 128 tile stores element by element (a quantisation word per column, raw accumulators, atomic
    additions) run on a kernel that does not, where both are candidates; the whole numbers are exact."""
    gen = torch.Generator(device="cuda").manual_seed(n)
    a, b = (torch.randint(-8, 9, (x, k), generator=gen, device="cuda", dtype=torch.int8) for x in (m, n))
    acc = (a.double() @ b.double().t()).to(torch.int32)
    if drain == "column words":  # scale 2^-4, no offset, signed bytes
        words = torch.full((n,), (int(np.float32(2.0 ** -4).view(np.uint32)) & 0xFFFFE000) | (1 << 46), dtype=torch.int64, device="cuda")
        got = pa.gemm_requant(a, b, pa.I8, pa.I8, words, per_column=True)
        ref = torch.round(acc.double() / 16).clamp(-128, 127).to(torch.int8)
    elif drain == "raw":
        ones = torch.ones(max(m, n), device="cuda")
        got, ref = pa.gemm_w8a8(a, b, ones[:m], ones[:n], want_acc=True)[1], acc
    else:
        got = torch.ones((m, n), device="cuda")
        pa.gemm_atomic_add(got, a.bfloat16(), b.bfloat16(), pa.BF16)
        ref = acc.float() + 1
    assert not pa.last_kernel().startswith("tile128x128_dtl"), pa.last_kernel()
    assert torch.equal(got, ref)


@pytest.mark.parametrize("kind,m,n,k,pitch,kernel", [
    ("bf16", 117, 888, 49, 49, "tile64x64_bf16"), ("bf16", 1609, 448, 280, 281, "tile64x64_bf16"), ("bf16", 4633, 10496, 512, 513, "tile128x128_bf16"),
    ("bf16", 125, 2624, 64, 64, "tile64x64_bf16"), ("i8", 69, 68, 34, 34, "tile64x64_i8"), ("i8", 1609, 448, 560, 561, "tile64x64_i8"),
    ("bf16", 64, 4097, 4095, 4095, "tile64x64_any_bf16"), ("bf16", 125, 2624, 1024, 1024, "tile64x32_dtl_bf16")])
def test_short_k_runs_on_the_register_staged_tiles(pa, kind, m, n, k, pitch, kernel):  # noqa: F811
    """A few slabs of K, rows on any byte (odd K; whole chunks of K at an odd pitch) and aligned, keep the register-staged tiles;
    longer ones take the deep-ring kernel.  Exact products of small whole numbers."""
    tdt, t, tc = (torch.int8, pa.I8, pa.I32) if kind == "i8" else (torch.bfloat16, pa.BF16, pa.F32)
    gen = torch.Generator(device="cuda").manual_seed(k)
    a, b = (torch.randint(-3, 4, (x, pitch), generator=gen, device="cuda").to(tdt) for x in (m, n))
    got = pa.gemm(a, b, t, tc, pa.B_DN, k=k)
    assert pa.last_kernel() == kernel, pa.last_kernel()
    assert torch.equal(got.double(), a[:, :k].double() @ b[:, :k].double().t())


def test_short_k_block_scaled_products_run_on_the_register_staged_tile(pa, oracle):  # noqa: F811
    r = np.random.default_rng(3)
    m, n, k = 105, 256, 256
    a, b, sa, sb = _mx_inputs(r, ob.E2M1, m, n, k)
    got = host(pa.gemm_mx(dev(a), dev(b), dev(sa), dev(sb), m, n, k, pa.E2M1, pa.E2M1, pa.F32))
    assert pa.last_kernel() == "tile64x64_fp4_e2m1", pa.last_kernel()
    assert relerr(got, oracle.matmul_mx(a, b, sa, sb, m, k, n, ob.E2M1, ob.E2M1)) <= 1e-4


@pytest.mark.parametrize("m,n,k,scales", [(943, 22144, 96, False), (1536, 12416, 384, True), (1536, 12416, 644, True), (4096, 4312, 64, False)])
def test_tail_columns_on_either_kernel(pa, m, n, k, scales):  # noqa: F811
    """Tail columns of a 256 x 256 grid that make more than a round of 128 x 128 tiles, W8A8 ones below and above the K from which
    the deep-ring kernel takes them, and a narrow last column: the bits of the single launch."""
    gen = torch.Generator(device="cuda").manual_seed(k)
    if scales:
        a, b = (torch.randint(-128, 128, (x, k), generator=gen, device="cuda", dtype=torch.int8) for x in (m, n))
        sa, sb = (torch.rand(x, generator=gen, device="cuda") for x in (m, n))
        run = lambda: pa.gemm_w8a8(a, b, sa, sb)  # noqa: E731
    else:  # whole numbers: exact in any order
        a, b = (torch.randint(-7, 8, (x, k), generator=gen, device="cuda").to(torch.bfloat16) for x in (m, n))
        run = lambda: pa.gemm(a, b, pa.BF16, pa.F32, pa.B_DN)  # noqa: E731
    got = run()
    assert pa.last_kernel().startswith("tile256x256w8_dtl"), pa.last_kernel()
    with tile_env(PTOAMD_NO_TAIL_SPLIT="1"):
        assert torch.equal(got, run())


@pytest.mark.parametrize("m,n,k,kernel", [(640, 22848, 192, "tile192x128_bnd_bf16"), (640, 22848, 384, "tile192x128_bnd_bf16"), (640, 22848, 1024, "tile256x256w8_bnd_bf16"),
                                          (4000, 4288, 64, "tile256x256w8_bnd_bf16")])
def test_row_major_b_short_k_off_the_256x256_tile(pa, m, n, k, kernel):  # noqa: F811
    """A round of 256 x 256 tiles from a row-major B: below 512 elements of K the other kernels compete for it where more than a
    tenth of those tiles lies past the matrix."""
    gen = torch.Generator(device="cuda").manual_seed(k)
    a, b = (torch.randint(-3, 4, x, generator=gen, device="cuda").to(torch.bfloat16) for x in ((m, k), (k, n)))
    got = pa.gemm(a, b, pa.BF16, pa.F32, pa.B_ND)
    assert pa.last_kernel() == kernel, pa.last_kernel()
    assert torch.equal(got.double(), a.double() @ b.double())


@pytest.mark.parametrize("kind,m,n,k,kernel", [("bf16", 1391, 9546, 6800, "tile256x256w8_dtl_bf16"), ("i8", 2117, 5492, 9300, "tile256x256w8_dtl_i8"),
                                               ("bf16", 1237, 4100, 2056, "tile192x128_dtl_bf16"), ("bf16", 3044, 3712, 2392, "tile192x128_dtl_bf16")])
def test_long_k_off_the_lines(pa, kind, m, n, k, kernel):  # noqa: F811
    """A long K that is no whole number of slabs, on a grid that nearly fills the chip, runs on the 256 x 256 tile, a smaller grid
    on the deep-ring kernel.  Exact products of small whole numbers."""
    tdt, t, tc = (torch.int8, pa.I8, pa.I32) if kind == "i8" else (torch.bfloat16, pa.BF16, pa.F32)
    gen = torch.Generator(device="cuda").manual_seed(k)
    a, b = (torch.randint(-3, 4, (x, k), generator=gen, device="cuda").to(tdt) for x in (m, n))
    got = pa.gemm(a, b, t, tc, pa.B_DN)
    assert pa.last_kernel() == kernel, pa.last_kernel()
    assert torch.equal(got.double(), a.double() @ b.double().t())


@pytest.mark.parametrize("m,n,k,per_column", [(2914, 4275, 256, False), (2504, 5006, 384, False), (2256, 6604, 768, True)])
def test_requantised_columns_that_end_inside_a_wave_tile(pa, m, n, k, per_column):  # noqa: F811
    """The 256 x 256 tile, which stores such columns as it does whole wave tiles, where it is ahead; the bits of a smaller tile."""
    gen = torch.Generator(device="cuda").manual_seed(k)
    a, b = (torch.randint(-99, 100, (x, k), generator=gen, device="cuda", dtype=torch.int8) for x in (m, n))
    words = ((torch.rand(n if per_column else 1, generator=gen, device="cuda") * 1e-4 + 1e-4).view(torch.int32).to(torch.int64) & 0xFFFFE000) | (1 << 46)
    got = pa.gemm_requant(a, b, pa.I8, pa.I8, words, per_column=per_column)
    assert pa.last_kernel() == "tile256x256w8_dtl_i8", pa.last_kernel()
    with tile_env(PTOAMD_TILE=2):
        assert torch.equal(got, pa.gemm_requant(a, b, pa.I8, pa.I8, words, per_column=per_column))
    assert got.unique().numel() > 100


@pytest.mark.parametrize("shape", range(9))
@pytest.mark.parametrize("kind", ["bf16", "i8", "fp8"])
def test_every_count_of_stages(pa, kind, shape):  # noqa: F811
    """One stage of K to three more than a ring holds, whole and with a chunk and four bytes more (fp8: MX blocks), every remainder of a
    thread's columns, 32- and 16-bit results: exact, the sums being whole numbers below 2^24."""
    scaled = kind == "fp8"
    if scaled and SHAPES[shape][3] is None:
        pytest.skip("the plain types' shape")
    bm, bn, stage = SHAPES[shape][0], SHAPES[shape][1], SHAPES[shape][3 if scaled else 2]
    gen = torch.Generator(device="cuda").manual_seed(shape)
    for count in range(1, 8):
        for tail in (0, 128 if scaled else 20):
            kb, m, n = count * stage + tail, bm + 1, bn + count
            k = kb // 2 if kind == "bf16" else kb
            a, b = (torch.randint(-3, 4, (x, k), generator=gen, device="cuda") for x in (m, n))
            ref = a.double() @ b.double().T
            with tile_env(PTOAMD_RING=shape):
                if kind == "fp8":
                    lut = torch.tensor([0, 0x38, 0x40, 0x44], device="cuda", dtype=torch.uint8)  # 0, 1, 2, 3 in E4M3
                    ca, cb = (lut[x.abs()] | (0x80 * (x < 0)).to(torch.uint8) for x in (a, b))
                    got = pa.gemm_fp8(ca, cb, pa.E4M3, pa.E4M3, pa.F32 if count % 2 else pa.BF16)
                elif kind == "bf16":
                    bias = torch.randint(-9, 10, (n,), generator=gen, device="cuda").float()
                    got = pa.gemm(a.bfloat16(), b.bfloat16(), pa.BF16, pa.F32 if count % 2 else pa.BF16, pa.B_DN, bias=bias)
                    ref = ref + bias.double()
                else:
                    got = pa.gemm(a.to(torch.int8), b.to(torch.int8), pa.I8, pa.I32, pa.B_DN)
                assert pa.last_kernel().startswith(f"tile{bm}x{bn}_"), pa.last_kernel()
            assert torch.equal(got, ref.float().to(got.dtype)), (kind, m, n, kb)


@pytest.mark.parametrize("kind,shape", [("bf16", s) for s in range(9)] + [("fp8", s) for s in range(7)])
def test_last_group_of_tile_rows(pa, kind, shape):  # noqa: F811
    """One, two and three tile rows behind whole groups of four, several tile columns: exact, the sums being whole numbers."""
    bm, bn = SHAPES[shape][:2]
    gen = torch.Generator(device="cuda").manual_seed(shape)
    lut = torch.tensor([0, 0x38, 0x40, 0x44], device="cuda", dtype=torch.uint8)  # 0, 1, 2, 3 in E4M3
    for rest in (1, 2, 3):
        m, n, k = (8 + rest) * bm - 3, 5 * bn - 7, 128
        a, b = (torch.randint(-3, 4, (x, k), generator=gen, device="cuda") for x in (m, n))
        with tile_env(PTOAMD_RING=shape):
            if kind == "fp8":
                got = pa.gemm_fp8(*(lut[x.abs()] | (0x80 * (x < 0)).to(torch.uint8) for x in (a, b)), pa.E4M3, pa.E4M3, pa.F32)
            else:
                got = pa.gemm(a.bfloat16(), b.bfloat16(), pa.BF16, pa.F32, pa.B_DN)
            assert pa.last_kernel().startswith(f"tile{bm}x{bn}_"), pa.last_kernel()
        assert torch.equal(got.double(), a.double() @ b.double().T), (m, n)


@pytest.mark.parametrize("shape", [1, 3, 4, 5, 6, 7, 8])
def test_row_major_b_rows_on_any_element_through_every_drain(pa, shape):  # noqa: F811
    """As above with a bias row and a 16-bit result, an accumulator input, a quantisation word for all columns and one per column, atomic
    additions: exact, the sums being whole numbers; what is quantised as on the order-exact kernel."""
    bm, bn, stage = SHAPES[shape][:3]
    gen = torch.Generator(device="cuda").manual_seed(shape)
    m, n, k = bm + 1, bn + 3, 2 * (stage // 2) + 5
    a, b = (torch.randint(-3, 4, x, generator=gen, device="cuda").bfloat16() for x in ((m, k), (k, n)))
    ref = a.double() @ b.double()
    bias = torch.randint(-9, 10, (n,), generator=gen, device="cuda").float()
    c_in = torch.randint(-9, 10, (m, n), generator=gen, device="cuda").float()
    words = ((torch.randint(0, 2 ** 5, (n,), generator=gen, device="cuda") << 37) | (torch.arange(n, device="cuda") % 2 * (1 << 46))) | 0x3E000000
    name = f"tile{bm}x{bn}_bnd_any_bf16"
    with tile_env(PTOAMD_RING=shape):
        got = pa.gemm(a, b, pa.BF16, pa.BF16, pa.B_ND, bias=bias)
        assert pa.last_kernel() == name and torch.equal(got, (ref + bias.double()).float().bfloat16())
        assert torch.equal(pa.gemm(a, b, pa.BF16, pa.F32, pa.B_ND, c_in=c_in).double(), ref + c_in.double())
        c = c_in.clone()
        pa.gemm_atomic_add(c, a, b, pa.BF16, pa.B_ND)
        assert pa.last_kernel() == name and torch.equal(c.double(), ref + c_in.double())
        quantised = [pa.gemm_requant(a, b, pa.BF16, t, w, per_column=w.numel() > 1, b_layout=pa.B_ND) for t in (pa.I8, pa.F16) for w in (words[:1].contiguous(), words)]
        assert pa.last_kernel() == name
    with tile_env(PTOAMD_FORCE_GENERIC=1):
        exact = [pa.gemm_requant(a, b, pa.BF16, t, w, per_column=w.numel() > 1, b_layout=pa.B_ND) for t in (pa.I8, pa.F16) for w in (words[:1].contiguous(), words)]
    for q, e in zip(quantised, exact):
        assert torch.equal(q, e) and q.unique().numel() > 10
