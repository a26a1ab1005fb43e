"""What the package's Makefile rebuilds (no compiler is run)."""
import os
import shutil
import subprocess

MAKEFILE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "pto-isa-mirror_amd", "Makefile")


def test_changed_flags_rebuild_everything(tmp_path):
    """The flags stand in the Makefile: what was built before it changed is built again, also the objects with flags of their own."""
    shutil.copy(MAKEFILE, tmp_path)
    sources = ["csrc/quant.hip", "csrc/gemm_ring_bf16.hip", "csrc/gemm_tile_bf16.hip", "kernels/gemm_tiled.hip"]
    targets = ["build/quant.o", "build/gemm_ring_bf16.o", "build/gemm_tile_bf16.o", "lib/libpto_gemm_tiled.so", "lib/libptoamd.so"]
    for age, names in ((0, sources + ["Makefile"]), (100, targets[:3]), (200, targets[3:])):
        for name in names:
            path = tmp_path / name
            path.parent.mkdir(exist_ok=True)
            path.touch()
            os.utime(path, (1_000_000_000 + age,) * 2)

    def commands():
        return subprocess.run(["make", "-n", "HIPCC=hipcc", "PYTHON=false"] + targets, cwd=tmp_path, check=True, capture_output=True, text=True).stdout.splitlines()

    assert not [c for c in commands() if c.startswith("hipcc")]
    os.utime(tmp_path / "Makefile", (1_000_000_300,) * 2)
    built = [c for c in commands() if c.startswith("hipcc")]
    for name in targets:
        assert any(f"-o {name}" in c for c in built), (name, built)
    assert "-amdgpu-kernarg-preload-count=14" in next(c for c in built if "-o build/quant.o" in c)
