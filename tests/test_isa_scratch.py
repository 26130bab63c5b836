"""CPU-side check of the code generated for gfx950: no kernel keeps registers in scratch memory.

A spill in a loop costs its traffic, and scratch accesses share the vector-memory counter by which the kernels wait for
their tile copies.  One instantiation is known to: the split schedule under an additive bias."""
import os
import re
import shutil
import subprocess

import pytest

from mojodiffusion_amd import _lib

READELF = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin", "llvm-readelf")
OBJDUMP = os.path.join(os.path.dirname(READELF), "llvm-objdump")
KNOWN = {"_ZN4sage16sage_attn_kernelILi128ELi0ELb0ELb1ELb1E": 20}       # prefix: bytes per lane


@pytest.mark.skipif(not (os.path.exists(READELF) and os.path.exists(OBJDUMP)), reason="no LLVM tools")
def test_no_kernel_spills(tmp_path):
    copy = shutil.copy(_lib.LIB_PATH, tmp_path)         # (the bundles are written next to the input)
    subprocess.run([OBJDUMP, "--offloading", copy], check=True, stdout=subprocess.DEVNULL)
    scratch = {}
    for name in sorted(os.listdir(tmp_path)):
        if name.endswith("gfx950"):
            text = subprocess.run([READELF, "--notes", os.path.join(tmp_path, name)], check=True, capture_output=True, text=True).stdout
            for symbol, size in re.findall(r"\.name:\s+(_Z\S+).*?\.private_segment_fixed_size:\s+(\d+)", text, re.S):
                scratch[symbol] = int(size)
    assert len(scratch) > 80
    over = {s: n for s, n in scratch.items() if n > max((b for p, b in KNOWN.items() if s.startswith(p)), default=0)}
    assert not over, over
