"""CPU check of the built library's kernel metadata: no kernel uses scratch memory.

A spilled register is a round trip to memory beside the kernel's own traffic, and every
kernel's registers are budgeted to fit.
"""

import glob
import os
import re
import shutil
import subprocess

import pytest

LLVM = "/opt/rocm/llvm/bin"


@pytest.mark.skipif(not os.path.exists(f"{LLVM}/llvm-readelf"), reason="needs the ROCm toolchain")
def test_no_kernel_uses_scratch(tmp_path):
    from cobra_amd import _lib

    shutil.copy(_lib.LIB_PATH, tmp_path / "lib.so")
    subprocess.run([f"{LLVM}/llvm-objdump", "--offloading", "lib.so"], cwd=tmp_path, check=True, capture_output=True)
    kernels, scratch = 0, []
    for obj in glob.glob(str(tmp_path / "*gfx950*")):
        notes = subprocess.run([f"{LLVM}/llvm-readelf", "--notes", obj], check=True, capture_output=True,
                               text=True).stdout
        for name, size in re.findall(r"\.name: +(\S+)\n +\.private_segment_fixed_size: (\d+)", notes):
            kernels += 1
            if int(size):
                scratch.append((name, int(size)))
    assert kernels > 100
    assert not scratch, scratch
