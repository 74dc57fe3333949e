"""The tile GEMM kernels, compiled for the GPU, keep everything in registers and LDS: with a few registers spilled in a path
that hardly any call takes, every launch of the kernel pays for scratch memory."""
import os
import re
import shutil
import subprocess

import pytest

LIB = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "fp-quant_amd", "fp_quant", "_lib", "libfpq_hip.so")
BIN = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin")


needs_build = pytest.mark.skipif(not os.path.exists(LIB) or not os.path.exists(os.path.join(BIN, "llvm-readelf")),
                                 reason="needs the built library and the compiler's llvm-readelf")


def private_segments(tmp_path):
    shutil.copy(LIB, tmp_path / "lib.so")
    subprocess.run([os.path.join(BIN, "llvm-objdump"), "--offloading", "lib.so"], cwd=tmp_path, check=True, capture_output=True)
    sizes = {}
    for name in os.listdir(tmp_path):
        if "gfx950" in name:
            notes = subprocess.run([os.path.join(BIN, "llvm-readelf"), "--notes", name], cwd=tmp_path, check=True,
                                   capture_output=True, text=True).stdout
            for kernel, size in re.findall(r"\.name: +(_Z\S+)\n(?:(?!\.name:).)*?\.private_segment_fixed_size: (\d+)", notes, re.S):
                sizes[kernel] = int(size)
    return sizes


@needs_build
def test_tile_gemm_kernels_use_no_scratch(tmp_path):
    sizes = private_segments(tmp_path)
    tiles = {k: v for k, v in sizes.items() if "gemm_fp4_packed_kernel" in k}
    assert len(tiles) >= 10 and not any(tiles.values()), {k: v for k, v in tiles.items() if v}


@needs_build
def test_streaming_gemm_and_tile_quantizer_use_no_scratch(tmp_path):
    sizes = private_segments(tmp_path)
    found = {k: v for k, v in sizes.items() if "gemm_fp4_stream_kernel" in k or re.match(r"_ZN3fpq\d+tile_quantize_kernel", k)}
    # one form keeps three registers there: NVFP4, 128-wide rotation, SiLU*up over a ragged K
    spills = {k: v for k, v in found.items() if v > (12 if "20tile_quantize_kernelILi128ELi1ELi0ELi1ELi2ELb0ELb1EE" in k else 0)}
    assert len(found) >= 200 and not spills, spills
