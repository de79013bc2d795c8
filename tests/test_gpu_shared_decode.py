"""k_huf_mmv with several columns per decode (dense products of the reference's layouts): every column has the bits of its
single-column launch, at every column count, in both formats and chunk orders, with a ragged last block and column group."""
from __future__ import annotations

import pytest
import torch

from orin_qwen_lossless_amd import synth
from test_gpu_kernels import HP, HUF, enc, tbf16

pytestmark = pytest.mark.gpu


# units around 8 and 16 per CU (a column by itself, two, four) and beyond; the most columns of LDS (K = 4096)
@pytest.mark.parametrize("fmt,K,R,units,cm", [(HP, 512, 1, 1025, False), (HP, 512, 1, 2049, False), (HP, 1024, 4, 2051, True), (HP, 1536, 2, 1031, False),
                                              (HP, 2048, 8, 525, False), (HP, 4096, 1, 2051, False), (HP, 2048, 8, 1030, True),
                                              (HUF, 512, 1, 2051, False), (HUF, 1536, 4, 1030, False), (HUF, 4096, 1, 2051, False)])
def test_columns_that_share_a_decode(ops, fmt, K, R, units, cm):
    rows = R * units
    w = enc(ops, synth.weights(rows, K, rows + K), fmt, R, cm, False)
    x = tbf16(synth.activations(11, K, 7))
    for xt in (x, x.float()):
        one = torch.cat([ops.mmv(xt[t:t + 1], w) for t in range(11)])
        for t in (2, 3, 4, 5, 7, 8, 11):
            assert torch.equal(ops.mmv(xt[:t], w), one[:t]), t
        assert torch.equal(ops.mmv(xt[:7], w, out_dtype=torch.bfloat16), one[:7].to(torch.bfloat16))
    wide = torch.zeros((5, K + 64), dtype=x.dtype, device="cuda")
    wide[:, :K] = x[:5]
    assert torch.equal(ops.mmv(wide[:, :K], w), ops.mmv(x[:5], w))
