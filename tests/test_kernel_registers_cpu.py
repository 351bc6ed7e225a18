"""Registers of the built kernels whose waves in flight hang on a few of them: read from the notes of the code object."""

import os
import re
import subprocess

import pytest

from async_llm_amd import build

LLVM = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin")
BUNDLE = os.path.join(build.OBJ_DIR, "viewattn.hipfb")
LANE_REGISTERS = 512  # of a SIMD, per lane


@pytest.mark.skipif(not (os.path.exists(BUNDLE) and os.path.exists(os.path.join(LLVM, "llvm-readelf"))),
                    reason="needs the objects of a build and the LLVM tools")
def test_fp32_vector_kernel_leaves_room_for_four_waves(tmp_path):
    elf = str(tmp_path / "viewattn.elf")
    subprocess.run([os.path.join(LLVM, "clang-offload-bundler"), "--unbundle", "--type=o", "--input=" + BUNDLE,
                    "--targets=hipv4-amdgcn-amd-amdhsa--gfx950", "--output=" + elf], check=True)
    notes = subprocess.run([os.path.join(LLVM, "llvm-readelf"), "--notes", elf], check=True, capture_output=True,
                           text=True).stdout
    kernels = re.findall(r"\.name:\s+(\S*attn_generic_kernelINS_3F32E\S*)(.*?)\.vgpr_count:\s+(\d+)", notes, re.S)
    assert len(kernels) == 5  # head dims 16 to 256
    for name, between, registers in kernels:
        assert int(registers) * 4 <= LANE_REGISTERS, name
        assert re.search(r"\.private_segment_fixed_size:\s+0\b", between), name
