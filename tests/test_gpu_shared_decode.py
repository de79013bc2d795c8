"""k_huf_mmv with several columns per decode (dense products of the reference's layouts): every column has the bits of its
single-column launch, at every column count, in both formats and chunk orders, with a ragged last block and column group."""
from __future__ import annotations

import pytest
import torch

from orin_qwen_lossless_amd import synth
from test_gpu_kernels import HP, HUF, enc, tbf16

pytestmark = pytest.mark.gpu


reached: set[str] = set()


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
        assert ops.last_kernel().endswith(", 1>")
        for t in (2, 3, 4, 5, 7, 8, 11):
            assert torch.equal(ops.mmv(xt[:t], w), one[:t]), t
            reached.add(ops.last_kernel().split("<")[1][0] + ops.last_kernel()[-5:])
        assert torch.equal(ops.mmv(xt[:7], w, out_dtype=torch.bfloat16), one[:7].to(torch.bfloat16))
    if (fmt, K, units) == (HUF, 4096, 2051):                   # (the last case) every instance with rings
        assert reached >= {f"{f}1, {n}>" for f in (HP, HUF) for n in (1, 2, 3, 4)}, reached
    wide = torch.zeros((5, K + 64), dtype=x.dtype, device="cuda")
    wide[:, :K] = x[:5]
    assert torch.equal(ops.mmv(wide[:, :K], w), ops.mmv(x[:5], w))


# the lines between the instances on 256 CUs, for each count of columns: a last group of four with a column or two missing, four FP32
# columns of 4096 (a block per CU), pairs whose blocks fit the CUs at once, and both sides of the lines of single columns (15, 16 and 24
# half-waves per CU) and of fours (eight groups)
@pytest.mark.parametrize("fmt,K,R,units,f32,want", [
    (HP, 1024, 4, 1030, False, {3: 1, 4: 2, 5: 2, 7: 3, 8: 3, 10: 4}),
    (HP, 512, 1, 1024, False, {5: 1, 6: 1, 7: 2, 8: 2}),
    (HP, 512, 1, 1400, False, {4: 1, 5: 3, 7: 4, 9: 3}),
    (HP, 4096, 1, 1030, True, {3: 1, 5: 2, 7: 3, 10: 2, 12: 4}),
    (HP, 4096, 1, 2048, False, {2: 1, 3: 3, 4: 2}),
    (HP, 3072, 8, 1280, False, {2: 1, 3: 1, 4: 2}),
    (HP, 3072, 8, 1281, False, {2: 1, 3: 3, 4: 2}),
    (HUF, 4096, 1, 1400, True, {2: 1, 3: 3, 4: 2, 8: 2, 12: 3, 16: 4}),
    (HUF, 4096, 4, 800, True, {5: 1, 6: 3, 8: 2, 12: 3, 16: 4}),
    (HP, 512, 1, 9000, True, {1: 1, 2: 2, 3: 3, 4: 4, 5: 3, 9: 3}),
    (HUF, 512, 1, 9000, False, {2: 2, 5: 3, 8: 4})])
def test_the_instance_for_a_count_of_columns(ops, fmt, K, R, units, f32, want):
    if ops.cu_count() != 256:
        pytest.skip("the counts are those of 256 CUs")
    w = enc(ops, synth.weights(R * units, K, R * units + K), fmt, R, False, False)
    x = tbf16(synth.activations(16, K, 7))
    x = x.float() if f32 else x
    one = torch.cat([ops.mmv(x[t:t + 1], w) for t in range(16)])
    for t, nc in want.items():
        assert torch.equal(ops.mmv(x[:t], w), one[:t]), t
        assert ops.last_kernel() == f"k_huf_mmv<{fmt}, {'float' if f32 else 'bf16_t'}, 0, 1, {nc}>", t
