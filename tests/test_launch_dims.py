"""Launch shapes (csrc/launch_dims.h, no GPU code): no CU gets more wavefronts than an even split gives."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.skipif(shutil.which("g++") is None, reason="no g++")
def test_wavefronts_are_spread_over_the_device(tmp_path):
    exe = str(tmp_path / "launch_dims")
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-fsanitize=undefined", "-fno-sanitize-recover=undefined",
                    "-I" + os.path.join(ROOT, "orin_qwen_lossless_amd", "csrc"), os.path.join(ROOT, "tests", "cpp", "launch_dims.cpp"), "-o", exe],
                   check=True, capture_output=True, timeout=120)
    out = subprocess.run([exe], check=True, capture_output=True, text=True, timeout=60).stdout.splitlines()
    for ln, (cus, full) in zip(out, [(c, f) for c in (256, 64, 1) for f in (8, 16)]):
        head, values = ln.split(": ")
        over, largest, filled = map(int, values.split())
        assert head == f"{cus} {full}" and over == 0 and largest <= 16 and filled == full, ln
    assert out[-1] == "9 9 8"
