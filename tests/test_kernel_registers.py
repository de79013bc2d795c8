"""Kernels whose launches count on eight wavefronts to a SIMD take no more than its 512 registers allow them: 64."""
from __future__ import annotations

import os
import re
import subprocess

import pytest

from orin_qwen_lossless_amd import build

LLVM = os.path.join(os.path.dirname(os.path.dirname(os.path.realpath(build.HIPCC))), "llvm", "bin")
OBJECT = os.path.join(build.OBJ, "kernels_compat.hip.o")


@pytest.mark.skipif(not (os.path.exists(OBJECT) and os.path.exists(os.path.join(LLVM, "clang-offload-bundler"))), reason="reads the objects of a build")
def test_the_4_bit_gemv_of_one_column_and_one_pair(tmp_path):
    fat, code = str(tmp_path / "fat"), str(tmp_path / "code")
    run = lambda tool, *args: subprocess.run([os.path.join(LLVM, tool), *args], check=True, capture_output=True, text=True).stdout  # noqa: E731
    run("llvm-objcopy", f"--dump-section=.hip_fatbin={fat}", OBJECT, os.devnull)
    run("clang-offload-bundler", "--type=o", "--unbundle", "--targets=hipv4-amdgcn-amd-amdhsa--gfx950", f"--input={fat}", f"--output={code}")
    notes = run("llvm-readelf", "--notes", code)
    found = {name: int(count) for name, count in re.findall(r"\.name:\s+(\S+)\n(?:(?!\.name:).)*?\.vgpr_count:\s+(\d+)", notes, re.S)}
    mine = {n: c for n, c in found.items() if re.search(r"k_nib_mmvI(f|NS0_6bf16_tE)Li[012]ELi1ELi1EEE", n)}
    assert len(mine) == 6 and max(mine.values()) <= 64, mine
