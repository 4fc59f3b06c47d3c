"""What the built kernels ask of a SIMD's 512 vector registers, where their speed rests on how many
waves share it (the code objects' own metadata; no GPU)."""
import re
import subprocess
from pathlib import Path

import pytest

OBJ = Path(__file__).resolve().parents[1] / "axon-infer_amd" / "csrc" / "_build" / "hip"
LLVM = Path("/opt/rocm/llvm/bin")


def kernels(name, tmp_path):
    """{kernel symbol: (vector registers, spilled ones)} of hip/<name>.hip."""
    obj = OBJ / f"{name}.o"
    if not obj.exists() or not (LLVM / "clang-offload-bundler").exists():
        pytest.skip("needs the built object and the ROCm toolchain")
    fat, code = tmp_path / "fat", tmp_path / "code"
    subprocess.run([str(LLVM / "llvm-objcopy"), f"--dump-section=.hip_fatbin={fat}", str(obj), str(tmp_path / "copy.o")], check=True)
    subprocess.run([str(LLVM / "clang-offload-bundler"), "--unbundle", "--type=o", f"--input={fat}", f"--output={code}",
                    "--targets=hipv4-amdgcn-amd-amdhsa--gfx950"], check=True)
    notes = subprocess.run([str(LLVM / "llvm-readelf"), "--notes", str(code)], check=True, capture_output=True, text=True).stdout
    out = {}
    for part in notes.split("- .agpr_count:")[1:]:
        value = lambda key: re.search(rf"\.{key}:\s+(\S+)", part).group(1)
        out[value("name")] = (int(value("vgpr_count")), int(value("vgpr_spill_count")))
    assert out
    return out


def test_two_tiled_attention_workgroups_fit_a_cu(tmp_path):
    """Eight waves each, so four per SIMD: at most 128 registers, with either cache type."""
    found = {k: v for k, v in kernels("attention", tmp_path).items() if re.search(r"attention_tile_kernelILb[01]E(Lj4ELj8|Lj8ELj4)E", k)}
    assert len(found) == 4
    for k, (registers, spilled) in found.items():
        assert registers <= 128 and spilled == 0, k
