"""Register allocation of the shipped kernels, read from the built library (no GPU needed).

A kernel that spills keeps part of its working set in scratch memory; for the tile GEMM kernels that has cost up to a
tenth of the run time without failing any result check, so the library's own code-object metadata is checked here:
no kernel of the library may use scratch at all.
"""
import os
import re
import struct
import subprocess

import msgpack
import pytest

LIB = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "pto-isa-mirror_amd", "lib", "libptoamd.so")
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _code_objects(blob):
    """Yield the gfx950 ELF images of every offload bundle in the shared library."""
    pos = blob.find(MAGIC)
    while pos >= 0:
        (count,) = struct.unpack_from("<Q", blob, pos + len(MAGIC))
        off = pos + len(MAGIC) + 8
        for _ in range(count):
            start, size, tlen = struct.unpack_from("<QQQ", blob, off)
            triple = blob[off + 24:off + 24 + tlen].decode()
            off += 24 + tlen
            if "amdgcn" in triple and size:
                assert triple.endswith("gfx950"), triple
                yield blob[pos + start:pos + start + size]
        pos = blob.find(MAGIC, pos + 1)


def _kernels(elf):
    """The amdhsa.kernels records of one code object (its NT_AMDGPU_METADATA note is a msgpack map)."""
    assert elf[:4] == b"\x7fELF" and elf[4] == 2, "64-bit ELF expected"
    shoff, = struct.unpack_from("<Q", elf, 0x28)
    shentsize, shnum = struct.unpack_from("<HH", elf, 0x3A)
    for i in range(shnum):
        sh_type, = struct.unpack_from("<I", elf, shoff + i * shentsize + 4)
        if sh_type != 7:  # SHT_NOTE
            continue
        off, size = struct.unpack_from("<QQ", elf, shoff + i * shentsize + 0x18)
        p, end = off, off + size
        while p + 12 <= end:
            namesz, descsz, ntype = struct.unpack_from("<III", elf, p)
            name = elf[p + 12:p + 12 + namesz].rstrip(b"\0")
            desc_at = p + 12 + (namesz + 3) // 4 * 4
            if name == b"AMDGPU" and ntype == 32:
                meta = msgpack.unpackb(elf[desc_at:desc_at + descsz], raw=False, strict_map_key=False)
                yield from meta.get("amdhsa.kernels", [])
            p = desc_at + (descsz + 3) // 4 * 4


@pytest.fixture(scope="module")
def kernels():
    if not os.path.exists(LIB):
        pytest.skip("libptoamd.so is not built")
    with open(LIB, "rb") as f:
        blob = f.read()
    ks = [k for elf in _code_objects(blob) for k in _kernels(elf)]
    assert ks, "no kernel metadata found in the library"
    return ks


def test_no_kernel_uses_scratch(kernels):
    names = [k[".name"] for k in kernels]
    for tag in ("gemm_tile_dtl_kernel", "gemm_tile_kernel", "gemv_mxfp4_splitk", "tquant_", "tdequant"):
        assert any(tag in n for n in names), (tag, names)
    spilled = {k[".name"]: k[".private_segment_fixed_size"] for k in kernels if k[".private_segment_fixed_size"]}
    assert not spilled, spilled


def test_large_tiles_keep_two_waves_per_simd(kernels):
    """The 8-wave 256 x 256 DMA tiles run two waves per SIMD: at most 256 vector registers, and an LDS budget set at
    launch (no static LDS)."""
    big = [k for k in kernels if "gemm_tile_dtl_kernel" in k[".name"] and "Li256ELi256ELi2ELi4" in k[".name"]]
    assert len(big) >= 8, [k[".name"] for k in kernels if "dtl" in k[".name"]]
    for k in big:
        assert k[".vgpr_count"] + k.get(".agpr_count", 0) <= 256, (k[".name"], k[".vgpr_count"], k.get(".agpr_count"))
        assert k[".max_flat_workgroup_size"] == 512


def test_register_staged_tiles_of_the_plain_types_share_a_simd(kernels):
    """Several workgroups of a register-staged tile run on a CU as long as its waves' registers let them: 128 x 128 tiles two waves
    a SIMD (their LDS admits two workgroups), 64 x 64 tiles four.  A SIMD has 512 registers per lane, given out by eights."""
    for edge, waves in (("Li128ELi128E", 2), ("Li64ELi64E", 4)):
        ks = [k for k in kernels if "16gemm_tile_kernel" in k[".name"] and edge in k[".name"] and any(op in k[".name"] for op in ("OpBF16", "OpF16", "OpI8"))]
        assert len(ks) >= 6, [k[".name"] for k in kernels if "gemm_tile_kernel" in k[".name"]]
        over = {k[".name"]: k[".vgpr_count"] for k in ks if (k[".vgpr_count"] + 7) // 8 * 8 * waves > 512}
        assert not over, over


def test_tiles_without_an_edge_carry_no_code_for_one(kernels):
    """Launches of whole wave tiles have kernels of their own (last template argument false) with no more registers than those that
    also store a wave tile that crosses N."""
    by_name = {k[".name"]: k[".vgpr_count"] for k in kernels if "gemm_tile_dtl_kernel" in k[".name"]}
    assert by_name
    for name, count in by_name.items():
        assert ("ELb0EEEv" in name) != ("ELb1EEEv" in name), name
        if "ELb1EEEv" in name:
            assert by_name[name.replace("ELb1EEEv", "ELb0EEEv")] <= count, name


def test_pipelined_deep_ring_tiles_hold_their_accumulators_once(kernels):
    """Deep-ring tiles of 64 x 64 to 128 x 128, copying waves beside multiplying ones: 16 to 64 accumulators a thread, two sets of
    fragments and, in the waves that copy rows on any byte, the pieces under way, all within a third of a SIMD's 512 registers.  A second
    set of accumulators for another copy of the K loop's code takes them past it.  (fp8 on 128 x 128 has fragments of twice the size.)"""
    shapes = ["64ELi64E", "96ELi64E", "128ELi64E", "128ELi128E"]
    ks = [k for k in kernels if "gemm_tile_ring_kernel" in k[".name"] and any(f"RingCfgILi{s}" in k[".name"] for s in shapes)]
    assert len(ks) >= 30, len(ks)
    over = {k[".name"]: k[".vgpr_count"] for k in ks if k[".vgpr_count"] > 168 and not ("OpFP8" in k[".name"] and "Li128ELi128E" in k[".name"])}
    assert not over, over


def test_rows_of_c_can_leave_either_way(tmp_path):
    """Tiles that store through LDS hold their 16-byte stores of C twice, non-temporal and plain, but for the result types that are never
    stored plainly.  The compiler can make one of two branches that differ in this only, then of plain stores, and no result would tell."""
    objdump = "/opt/rocm/llvm/bin/llvm-objdump"
    if not (os.path.exists(LIB) and os.path.exists(objdump)):
        pytest.skip("no library or no disassembler")
    with open(LIB, "rb") as f:
        blob = f.read()
    seen = 0
    for elf in _code_objects(blob):
        names = [k[".name"] for k in _kernels(elf) if "gemm_tile_dtl_kernel" in k[".name"] or "16gemm_tile_kernel" in k[".name"]]
        names = [n for n in names if "OpBF16" in n or "OpI8" in n]  # (the others are of the same templates)
        if not names:
            continue
        (tmp_path / "code.elf").write_bytes(elf)
        text = subprocess.run([objdump, "-d", "--no-show-raw-insn", "--disassemble-symbols=" + ",".join(names), str(tmp_path / "code.elf")],
                              check=True, capture_output=True, text=True).stdout
        for kernel in re.split(r"^[0-9a-f]+ <", text, flags=re.M)[1:]:
            stores = [line for line in kernel.splitlines() if "_store_dwordx4" in line]
            streamed = sum(" nt" in line for line in stores)
            assert 0 < len(stores) - streamed <= streamed, (kernel.split(">")[0], streamed, len(stores))
            seen += 1
    assert seen >= 20, seen
