"""k_nib_mmv with two (row, chunk) pairs per half-wave and k_nib_rows with several chunks in flight: the bits of launches
with one pair, every chunk count, row counts that end inside a block's second pair, escaped weights on both sides."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from orin_qwen_lossless_amd import synth
from test_gpu_kernels import NIB, bits, enc, tbf16

pytestmark = pytest.mark.gpu


# rows that make at least sixteen blocks per CU for one column (gate / up) and three (plain), and end at odd places
@pytest.mark.parametrize("K,rows", [(512, 32807), (1024, 16391), (1536, 8203), (2048, 8197), (2560, 4099), (3072, 4101), (3584, 4097), (4096, 4103)])
def test_two_pairs_have_the_bits_of_one(ops, K, rows):
    wb = synth.weights(rows, K, K + rows)
    for r, c in ((0, 3), (5, K - 1), (rows - 1, 7), (rows - 2, K // 2)):
        wb[r, c] = 0x4500                                    # an exponent outside the row's table
    w = enc(ops, wb, NIB)
    xb = synth.activations(3, K, 7)
    x, few = tbf16(xb), 64                                   # the first and last rows as matrices of their own: one pair
    ends = [(0, enc(ops, wb[:few], NIB)), (rows - few, enc(ops, wb[rows - few:], NIB))]
    for xt in (x, x.float()):
        y = ops.mmv(xt[:1], w)
        assert ops.last_kernel().endswith(", 0, 1, 2>")
        y3 = ops.mmv(xt, w, multi_col=False) if xt.dtype == torch.bfloat16 else ops.mmv(xt, w)
        glu = ops.mmv_glu2(xt[:1], w, w)
        assert ops.last_kernel().endswith(", 2, 1, 2>")
        for at, part in ends:
            ref = ops.mmv(xt[:1], part)
            assert ops.last_kernel().endswith(", 0, 1, 1>")
            assert torch.equal(y[:, at:at + few], ref)
            assert torch.equal(y3[:, at:at + few], torch.cat([ops.mmv(xt[t:t + 1], part) for t in range(3)]))
            assert torch.equal(glu[:, at:at + few], ops.mmv_glu2(xt[:1], part, part))
    assert np.array_equal(bits(ops.dequant(w)), wb)
    ids = torch.tensor([rows - 1, 0, 5, rows - 2], device="cuda")
    assert np.array_equal(bits(ops.get_rows(ids, w)), wb[ids.cpu().numpy()])
