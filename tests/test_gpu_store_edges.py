"""The staged store where a wave tile's columns reach past N: every element of C inside a wider buffer, nothing around it."""
import pytest
import torch

from test_gpu_parity import pa, tile_env  # noqa: F401

pytestmark = pytest.mark.gpu

# columns past the last whole 256, 128 or 64: each remainder of a 16-byte chunk, first and last columns of a wave tile
COLUMNS = [1, 2, 3, 63, 65, 100, 127, 132, 161, 254, 261]


def _product(pa, kind, a, b, out, bias, c_in):  # noqa: F811
    """The call, and what it has to give before the rounding to out's type: exact, all sums being small multiples of 1/4."""
    if kind == "w8a8":
        sa, sb = (2.0 ** -(torch.arange(x.shape[0], device="cuda") % 3).float() for x in (a, b))
        pa.gemm_w8a8(a.to(torch.int8), b.to(torch.int8), sa, sb, out=out)
        return (a.double() @ b.double().T) * sa.double()[:, None] * sb.double()
    if kind in ("fp8", "fp4"):
        m, k = a.shape
        table = {1: 2, 2: 4, 3: 5, 0: 0} if kind == "fp4" else {0: 0, 1: 0x38, 2: 0x40, 3: 0x44}
        sign = 8 if kind == "fp4" else 0x80

        def codes(x):
            lut = torch.tensor([table[i] for i in range(4)], device="cuda", dtype=torch.uint8)
            c = lut[x.abs().long()] | (sign * (x < 0)).to(torch.uint8)
            return (c[:, 0::2] | (c[:, 1::2] << 4)).contiguous() if kind == "fp4" else c
        ones = [torch.full((x.shape[0], k // 32), 127, dtype=torch.uint8, device="cuda") for x in (a, b)]
        t = pa.E2M1 if kind == "fp4" else pa.E4M3
        c_type = {torch.float32: pa.F32, torch.bfloat16: pa.BF16}[out.dtype]
        pa.gemm_mx(codes(a), codes(b), ones[0], ones[1], m, b.shape[0], k, t, t, c_type, out=out, c_in=c_in, bias=bias if c_in is None else None)
    else:
        tdt, t = {"bf16": (torch.bfloat16, pa.BF16), "f16": (torch.float16, pa.F16), "i8": (torch.int8, pa.I8)}[kind]
        c_type = {torch.float32: pa.F32, torch.bfloat16: pa.BF16, torch.float16: pa.F16, torch.int32: pa.I32}[out.dtype]
        pa.gemm(a.to(tdt), b.to(tdt), t, c_type, pa.B_DN, c_in=c_in, relu=c_in is not None, bias=bias, out=out)
    ref = a.double() @ b.double().T
    if c_in is not None:
        ref = ref + c_in.double()
    if bias is not None and not (kind in ("fp8", "fp4") and c_in is not None):
        ref = ref + bias.double()
    return ref.clamp_min(0) if c_in is not None and kind not in ("fp8", "fp4") else ref


@pytest.mark.parametrize("tile", [1, 2, 4, 5, 6, 7])
@pytest.mark.parametrize("kind,types", [("bf16", [torch.float32, torch.bfloat16]), ("f16", [torch.float16]), ("i8", [torch.int32]), ("w8a8", [torch.bfloat16]),
                                        ("fp8", [torch.bfloat16]), ("fp4", [torch.float32, torch.bfloat16])])
def test_wave_tiles_that_cross_n(pa, kind, types, tile):  # noqa: F811
    gen = torch.Generator(device="cuda").manual_seed(tile)
    for i, n in enumerate(COLUMNS):
        m, k, dtype = (1, 33, 129, 258)[i % 4], 512, types[i % len(types)]
        a, b = (torch.randint(-3, 4, (x, k), generator=gen, device="cuda") for x in (m, n))
        acc = torch.int32 if kind == "i8" else torch.float32
        bias = torch.randint(-9, 10, (n,), generator=gen, device="cuda").to(acc) if i % 3 == 1 and kind != "w8a8" else None
        lead = i % 3  # columns in front of C: its rows start on any element
        wide = torch.full((m, n + lead + 9), 77, device="cuda", dtype=dtype)
        # (the accumulator input has C's row pitch)
        c_in = torch.randint(-9, 10, wide.shape, generator=gen, device="cuda").to(acc)[:, lead:lead + n] if i % 3 == 2 and kind != "w8a8" else None
        with tile_env(PTOAMD_TILE=tile):
            ref = _product(pa, kind, a, b, wide[:, lead:lead + n], bias, c_in)
            name = pa.last_kernel()
        assert name.startswith("tile") and "ring" not in name, name
        # (one rounding: f32 and int32 hold the sums, the 16-bit types round what f32 holds)
        assert torch.equal(wide[:, lead:lead + n], ref.float().to(dtype)), (kind, tile, m, n, name)
        assert (wide[:, :lead] == 77).all() and (wide[:, lead + n:] == 77).all(), (kind, tile, m, n, name)


@pytest.mark.parametrize("tile", [1, 2, 4, 5, 6])
@pytest.mark.parametrize("kind", ["bf16", "i8"])
@pytest.mark.parametrize("per_column", [False, True])
def test_quantised_wave_tiles_that_cross_n(pa, per_column, kind, tile):  # noqa: F811
    """The same bits as the first columns of a product of whole tiles."""
    gen = torch.Generator(device="cuda").manual_seed(tile)
    tdt, t = (torch.bfloat16, pa.BF16) if kind == "bf16" else (torch.int8, pa.I8)
    names = {pa.I8: torch.int8, pa.U8: torch.uint8, pa.F16: torch.float16, pa.BF16: torch.bfloat16, pa.I16: torch.int16}
    m, k, most = 130, 256, 512
    a, b = (torch.randint(-3, 4, (x, k), generator=gen, device="cuda").to(tdt) for x in (m, most))
    scale = (torch.rand(most, generator=gen, device="cuda") * 0.5 + 0.25).view(torch.int32).to(torch.int64) & 0xFFFFE000
    words = scale | (torch.randint(0, 8, (most,), generator=gen, device="cuda") << 37) | (3 << 32)
    for i, n in enumerate(COLUMNS + [12, 77, 190]):
        c_type = [pa.I8, pa.U8, pa.F16, pa.I16 if kind == "i8" else pa.BF16][i % 4]
        signed = (1 << 46) if c_type == pa.I8 else 0
        q = (words if per_column else words[:1]) | signed
        wide = torch.full((m, n + 20), 77, device="cuda", dtype=names[c_type])
        lead = i % 3
        with tile_env(PTOAMD_TILE=tile):
            ref = pa.gemm_requant(a, b, t, c_type, q, per_column=per_column)
            pa.gemm_requant(a, b[:n], t, c_type, q[:n].contiguous(), per_column=per_column, out=wide[:, lead:lead + n])
        raw = torch.int8 if c_type in (pa.I8, pa.U8) else torch.int16
        assert torch.equal(wide[:, lead:lead + n].contiguous().view(raw), ref[:, :n].contiguous().view(raw)), (kind, tile, n, c_type)
        assert ref[:, :n].unique().numel() > 4
        assert (wide[:, :lead] == 77).all() and (wide[:, lead + n:] == 77).all(), (kind, tile, n, c_type)


@pytest.mark.parametrize("tile", [1, 2, 4, 5, 6])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_rows_on_and_off_the_64_byte_sectors(pa, dtype, tile):  # noqa: F811
    """Rows of C on whole sectors are stored non-temporally, others plainly: the same bits, nothing around them."""
    gen = torch.Generator(device="cuda").manual_seed(tile)
    m, n, k = 130, 261, 256
    a, b = (torch.randint(-3, 4, (x, k), generator=gen, device="cuda") for x in (m, n))
    ref = (a.double() @ b.double().T).float().to(dtype)
    sector = 64 // ref.element_size()
    wide = torch.empty(m * 400 + 2 * sector, device="cuda", dtype=dtype)
    assert wide.data_ptr() % 64 == 0
    # (row pitch in elements, columns in front of C): on the sectors; the pitch off them; the first row off them
    for pitch, lead in [(288, 0), (288, sector), (288 + sector // 2, 0), (289, 0), (288, 1), (288, sector // 2)]:
        wide.fill_(77)
        view = wide[:m * pitch].view(m, pitch) if lead == 0 else wide[lead:lead + m * pitch].view(m, pitch)
        with tile_env(PTOAMD_TILE=tile):
            pa.gemm(a.bfloat16(), b.bfloat16(), pa.BF16, pa.F32 if dtype == torch.float32 else pa.BF16, pa.B_DN, out=view[:, :n])
        assert torch.equal(view[:, :n], ref), (tile, pitch, lead)
        assert (view[:, n:] == 77).all() and (wide[:lead] == 77).all() and (wide[lead + m * pitch:] == 77).all(), (tile, pitch, lead)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.int32])
def test_rows_off_the_sectors_on_either_side_of_half_a_grid(pa, dtype):  # noqa: F811
    """127 tiles of 256 x 256, which stream them, and a row more, 128, which store them plainly."""
    gen = torch.Generator(device="cuda").manual_seed(1)
    n, k = 253, 64
    for m in (127 * 256, 127 * 256 + 1):
        a, b = (torch.randint(-3, 4, (x, k), generator=gen, device="cuda") for x in (m, n))
        if dtype == torch.int32:
            run = (a.to(torch.int8), b.to(torch.int8), pa.I8, pa.I32)
        else:
            run = (a.bfloat16(), b.bfloat16(), pa.BF16, pa.F32 if dtype == torch.float32 else pa.BF16)
        flat = torch.full((m * n + 1000,), 77, device="cuda", dtype=dtype)
        with tile_env(PTOAMD_TILE=4):
            pa.gemm(*run, pa.B_DN, out=flat[:m * n].view(m, n))
        assert torch.equal(flat[:m * n].view(m, n), (a.double() @ b.double().T).float().to(dtype)), m
        assert (flat[m * n:] == 77).all()


@pytest.mark.parametrize("tile", [1, 2, 4, 5, 6])
def test_requantised_rows_off_the_sectors_at_the_size_where_their_store_changes(pa, tile):  # noqa: F811
    """16-bit results by a word of 4 MiB less one row's and a row more."""
    gen = torch.Generator(device="cuda").manual_seed(tile)
    n, k = 1021, 64
    word = torch.tensor([0x3C000000], dtype=torch.int64, device="cuda")  # * 2 ** -7
    m0 = (4 << 20) // (2 * n)
    for m in (m0, m0 + 1):
        a, b = (torch.randint(-100, 100, (x, k), generator=gen, device="cuda", dtype=torch.int8) for x in (m, n))
        with tile_env(PTOAMD_TILE=tile):
            got = pa.gemm_requant(a, b, pa.I8, pa.F16, word, per_column=False)
        with tile_env(PTOAMD_FORCE_GENERIC=1):
            assert torch.equal(got, pa.gemm_requant(a, b, pa.I8, pa.F16, word, per_column=False)), (tile, m)
        assert got.unique().numel() > 100
