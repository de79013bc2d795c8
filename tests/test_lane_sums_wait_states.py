"""row_sums (csrc/dev_common.h) is inline asm, into which the compiler's hazard pass does not see: between a dot product and the
first add in there that reads its result stand three wait states, whatever the scheduler puts (or does not put) in between."""
from __future__ import annotations

import os
import re
import subprocess

import pytest

from conftest import ROOT
from orin_qwen_lossless_amd import build

SOURCE = """
#include "dev_common.h"
using namespace bf16n::dev;
// the dot products' operands are all there before the first of them, so that nothing is left to stand behind the last
__global__ void k(const uint32_t * p, float * y) {
    uint32_t w = p[threadIdx.x], x[COLS];
    float a[COLS];
    for (int i = 0; i < COLS; i++) {
        x[i] = p[64 * (i + 1) + threadIdx.x];
        a[i] = y[64 * (i + 1) + threadIdx.x];
    }
    __builtin_amdgcn_s_waitcnt(0);
    __builtin_amdgcn_sched_barrier(0);
    for (int i = COLS - 1; i >= 0; i--) { // (the sums begin with the last one's)
        a[i] = dot2_bf16(w, x[i], a[i]);
        __builtin_amdgcn_sched_barrier(0);
    }
    y[threadIdx.x] = row_sums<COLS>(a);
}
"""
WANTED = 3  # a VALU instruction that reads the result of v_dot2c_f32_bf16 (a DPP read of any VALU result: two)


@pytest.mark.parametrize("n", [1, 2, 3, 4])
def test_wait_states_between_dot_and_sum(tmp_path, n):
    src, out = tmp_path / "k.hip", tmp_path / "k.s"
    src.write_text(SOURCE)
    subprocess.run([build.HIPCC, *build.COMMON, *build.HIP_FLAGS, f"-DCOLS={n}", "--cuda-device-only", "-S", str(src), "-o", str(out)], check=True,
                   stderr=subprocess.DEVNULL, cwd=os.path.join(ROOT, "tests"))
    at, written, read = 0, {}, 0  # wait states so far; register -> where a dot product wrote it
    for line in out.read_text().splitlines():
        op, *args = re.split(r"[,\s]+", line.split(";")[0].strip())
        if not re.match(r"[sv]_|global_|ds_", op):
            continue
        sources = args[1:]
        if op.startswith("v_dot2"):
            written[args[0]] = at
        elif op.startswith("v_"):
            for r in sources:
                if r in written:
                    assert at - written.pop(r) - 1 >= WANTED, line
                    read += 1
        at += int(args[0], 0) + 1 if op == "s_nop" else 1
    assert read == n and not written
