"""The tile GEMM kernels, compiled for the GPU, keep everything in registers and LDS: with a few registers spilled in a path
that hardly any call takes, every launch of the kernel pays for scratch memory."""
import os
import re
import shutil
import subprocess

import pytest

LIB = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "fp-quant_amd", "fp_quant", "_lib", "libfpq_hip.so")
BIN = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin")


@pytest.mark.skipif(not os.path.exists(LIB) or not os.path.exists(os.path.join(BIN, "llvm-readelf")),
                    reason="needs the built library and the compiler's llvm-readelf")
def test_tile_gemm_kernels_use_no_scratch(tmp_path):
    shutil.copy(LIB, tmp_path / "lib.so")
    subprocess.run([os.path.join(BIN, "llvm-objdump"), "--offloading", "lib.so"], cwd=tmp_path, check=True, capture_output=True)
    sizes = {}
    for name in os.listdir(tmp_path):
        if "gfx950" in name:
            notes = subprocess.run([os.path.join(BIN, "llvm-readelf"), "--notes", name], cwd=tmp_path, check=True,
                                   capture_output=True, text=True).stdout
            for kernel, size in re.findall(r"\.name: +(_Z\S+)\n(?:(?!\.name:).)*?\.private_segment_fixed_size: (\d+)", notes, re.S):
                sizes[kernel] = int(size)
    tiles = {k: v for k, v in sizes.items() if "gemm_fp4_packed_kernel" in k}
    assert len(tiles) >= 10 and not any(tiles.values()), {k: v for k, v in tiles.items() if v}
