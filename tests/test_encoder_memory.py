"""Host memory of the wave64 encoder: beside the input and the two buffers it returns it holds a few blocks of units per
thread, not a second copy of the stream (0.35 byte per weight)."""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

CODE = """
import numpy as np, sys
from orin_qwen_lossless_amd import _lib, ops, synth

def peak():  # of this process image
    return next(int(ln.split()[1]) * 1024 for ln in open("/proc/self/status") if ln.startswith("VmHWM"))

rows, K, R = (int(v) for v in sys.argv[1:])
_lib.lib()
w = np.empty((rows, K), np.uint16)
part = synth.weights(512, K, 1)
for r in range(0, rows, 512):
    w[r:r + 512] = part
ops.encode_bits(part, 3, R, False, wave64=True)
before = peak()
plane, aux, fmt, unit = ops.encode_bits(w, 3, R, False, wave64=True)
assert (fmt, unit) == (3, R)
print((peak() - before - plane.nbytes - aux.nbytes) / (rows * K), aux.nbytes / (rows * K))
"""


@pytest.mark.skipif(not os.path.exists("/proc/self/status"), reason="no /proc")
@pytest.mark.parametrize("rows,K,R,scratch", [(65536, 2048, 16, 0.0), (131072, 512, 4, 0.0), (65536, 2048, 32, 2.0)])
def test_the_encoder_holds_the_stream_once(rows, K, R, scratch):
    """R = 32: the tile form encodes a permuted copy of the weights (two bytes each)."""
    out = subprocess.run([sys.executable, "-c", CODE, str(rows), str(K), str(R)], cwd=ROOT, check=True, capture_output=True, text=True, timeout=300)
    extra, aux = (float(v) for v in out.stdout.split())
    assert 0.3 < aux < 0.7
    # pages that the allocator keeps and the threads' blocks: a few MB of at least 67 M weights
    assert extra < scratch + 0.15, (extra, aux)
