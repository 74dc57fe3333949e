"""Kernels that ask for more dynamic LDS than a launch gets by itself: each has its limit raised, not only the first of a
launcher's (the state that remembers it is one per kernel in the built library)."""
import re
import shutil
import subprocess

import pytest

from fp_quant import _engine


@pytest.mark.skipif(not _engine.available() or shutil.which("nm") is None, reason="the library is not built, or no nm")
@pytest.mark.parametrize("kernel,which", [("rmsnorm_tile_quantize_kernel", r"I(\w*?)EEEv"),
                                          # (the packed one with the norm in front: ..., PACKED, PRO = RMSNorm, QUEST)
                                          ("quantize_stream_kernel", r"I(\w*?Lb1ELi1ELb0)EEEv")])
def test_every_kernel_of_a_launcher_has_its_limit_raised(kernel, which):
    names = subprocess.run(["nm", _engine.library_path()], capture_output=True, text=True, check=True).stdout.split()
    pattern = re.compile(rf"{kernel}{which}")
    kernels = {m[1] for n in names if n.startswith("_ZN3fpq") and (m := pattern.search(n))}
    raised = {m[1] for n in names if n.startswith("_ZZN3fpq15raise_lds_limit") and n.endswith("5limit")
              and (m := pattern.search(n))}
    assert len(kernels) > 1 and raised == kernels
