"""k_hp_split (HUFPAIR units whose lanes' streams are decoded in segments): the bits of the kernel with one half-wave per
unit, which takes the batches of more columns, for streams that fall into step, that never do, and of very short codes."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from orin_qwen_lossless_amd import synth
from test_gpu_kernels import HP, bits, enc, tbf16

pytestmark = pytest.mark.gpu


def _matrix(kind: str, rows: int, K: int) -> np.ndarray:
    wb = synth.weights(rows, K, rows + K)
    rng = np.random.default_rng(rows + K)
    if kind == "one":          # a single pair of exponents
        return np.full_like(wb, 0x3F81)
    if kind == "short":        # two exponents, one of them rare: codes of one bit, more of them in a segment than stay in registers
        return np.where(rng.random(wb.shape) < 0.03, 0x4081, 0x3F81).astype(np.uint16)
    if kind == "flat":         # 4096 pairs, equally frequent: codes of twelve bits throughout, which never fall into step
        return ((wb & 0x807F) | (rng.integers(64, 128, wb.shape) << 7)).astype(np.uint16)
    return wb


# one unit, more than a unit per CU and more than two, the fewest and the most pair codes a lane; both orders of the chunks
@pytest.mark.parametrize("kind,units,K,R,cm", [
    ("normal", 1, 2048, 16, False), ("normal", 300, 2048, 16, True), ("normal", 513, 2048, 16, False), ("normal", 5, 4096, 16, True),
    ("normal", 257, 4096, 16, False), ("normal", 33, 1024, 16, True), ("normal", 7, 2048, 8, False), ("normal", 9, 3072, 8, True),
    ("normal", 9, 2560, 8, False), ("one", 3, 2048, 16, False), ("short", 3, 2048, 16, False), ("short", 2, 4096, 16, True),
    ("flat", 3, 2048, 16, False), ("flat", 2, 4096, 16, False), ("flat", 2, 2048, 8, True)])
def test_split_units_have_the_bits_of_whole_ones(ops, kind, units, K, R, cm):
    rows = units * R
    wb = _matrix(kind, rows, K)
    w = enc(ops, wb, HP, R, cm, False)
    assert w.meta.format == HP and w.meta.chunk_major == cm
    xb = tbf16(synth.activations(9, K, 7))
    limit = min(8, (R * K // 64 - 128) // 48) if R * K // 64 <= 512 else 4
    for x in (xb, xb.float()):
        whole = ops.mmv(x, w)
        assert ops.last_kernel().startswith("k_huf_mmv") or ops.last_kernel() == ""
        for t in {1, 2, limit}:
            y = ops.mmv(x[:t], w)
            assert ops.last_kernel().startswith("k_hp_split<")
            assert torch.equal(y, whole[:t]), t
        assert torch.equal(ops.mmv(x[:1], w, out_dtype=torch.bfloat16), whole[:1].to(torch.bfloat16))
    assert np.array_equal(bits(ops.dequant(w)), wb)
    if units > 2:                                              # a range of units that ends before the matrix, and the last one
        assert np.array_equal(bits(ops.dequant(w, R, R)), wb[R:2 * R])
        assert np.array_equal(bits(ops.dequant(w, rows - R, R)), wb[-R:])
