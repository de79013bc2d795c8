"""k_w64_mmv_lds (several columns of 2048 or 4096, activations in LDS): every column has the bits of its single-column
launch."""
from __future__ import annotations

import pytest
import torch

from orin_qwen_lossless_amd import synth
from test_gpu_kernels import enc

pytestmark = pytest.mark.gpu


# one unit per wavefront (a single chain), two and a ragged end of three units (two chains, the second ends first); units of
# one loop body (a row) and of several
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("K,R,units", [(2048, 1, 64), (2048, 1, 8199), (4096, 1, 33), (4096, 1, 8199),
                                       (2048, 16, 37), (2048, 4, 4099), (4096, 16, 9), (4096, 2, 4099)])
def test_columns_in_lds_equal_single_columns(ops, K, R, units, dtype):
    rows = units * R
    w = enc(ops, synth.weights(rows, K, K + units), 3, R, False, True)
    x = synth.weights_torch(9, K, 5, "cuda").to(dtype)
    one = ops.mmv(x, w, multi_col=False)
    names = set()
    for t in range(1, 10):
        assert torch.equal(ops.mmv(x[:t], w), one[:t])
        names.add(ops.last_kernel().split("<")[0])
        y16 = ops.mmv(x[:t], w, out_dtype=torch.bfloat16)
        assert torch.equal(y16, one[:t].to(torch.bfloat16))
    assert "k_w64_mmv_lds" in names
