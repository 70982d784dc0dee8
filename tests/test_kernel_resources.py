"""What the compiler gave the kernels of every step (no GPU): none of them keeps registers in scratch memory. Read from the
notes of the code objects in the libraries as they are built here."""

import pathlib
import re
import subprocess

import pytest

import tie_amd  # noqa: F401
from tie_amd.kernels import build

READELF = pathlib.Path(build._hipcc()).resolve().parent.parent / "lib" / "llvm" / "bin" / "llvm-readelf"
if not READELF.exists():
    READELF = pathlib.Path("/opt/rocm/llvm/bin/llvm-readelf")


def scratch_bytes(tmp_path, name, source, defines=None):
    """Bytes of scratch a lane of every kernel of that library, by its mangled name."""
    data = build.compile_library(name, source, defines).read_bytes()
    found, at = {}, 1
    while (at := data.find(b"\x7fELF", at)) > 0:
        if data[at + 18:at + 20] != b"\xe0\x00":          # not a GPU's code object
            at += 4
            continue
        sections = int.from_bytes(data[at + 40:at + 48], "little")
        end = at + sections + int.from_bytes(data[at + 58:at + 60], "little") * int.from_bytes(data[at + 60:at + 62], "little")
        part = tmp_path / "code_object"
        part.write_bytes(data[at:end])
        notes = subprocess.run([str(READELF), "--notes", str(part)], capture_output=True, text=True, check=True).stdout
        for kernel in notes.split("- .agpr_count")[1:]:
            kernel_name = re.search(r"^\s+\.name:\s+(\S+)$", kernel, re.M)[1]
            found[kernel_name] = int(re.search(r"\.private_segment_fixed_size:\s+(\d+)", kernel)[1])
        at = end
    assert found, f"no kernels found in {name}"
    return found


@pytest.mark.skipif(not READELF.exists(), reason="no llvm-readelf here")
@pytest.mark.parametrize("name,source,kernels,count", [
    # the products that end a sub-layer: eight and sixteen waves
    ("tie_skinny_gemm_bf16", "skinny_gemm_bf16.hip", r"skinny_gemm_kernelILi1E.*Li(8|16)EEv", 8),
    ("tie_skinny_gemm_bf16", "skinny_gemm_bf16.hip", r"skinny_gemm_kernelILi[12]E.*Li4EEv", 96 + 48),
    ("tie_skinny_gemm_bf16", "skinny_gemm_bf16.hip", r"skinny_(half_tile|rows)_kernel", 4 + 12),
    # the norm of a sub-layer's result: up to eight values of a row a thread of 1024
    ("tie_elementwise", "elementwise.hip", r"norm_add_norm_row_kernel", 2 * (3 * 3 + 2)),
])
def test_kernels_without_scratch(tmp_path, name, source, kernels, count):
    scratch = {k: v for k, v in scratch_bytes(tmp_path, name, source).items() if re.search(kernels, k)}
    assert len(scratch) == count
    assert not [k for k, v in scratch.items() if v]


@pytest.mark.skipif(not READELF.exists(), reason="no llvm-readelf here")
@pytest.mark.parametrize("head_dim", [16, 64, 128, 256])
def test_the_ring_of_tiles_fits_the_registers(tmp_path, head_dim):
    """Decode attention holds tiles of keys in register sets that are loaded far ahead: as many as there is room for."""
    scratch = scratch_bytes(tmp_path, f"tie_attention_decode_bf16_hd{head_dim}", "attention_decode_bf16.hip",
                            {"HEAD_DIM": head_dim})
    ring = {k: v for k, v in scratch.items() if "attention_decode_ring_kernel" in k}
    assert len(ring) >= 3 and not [k for k, v in ring.items() if v]
