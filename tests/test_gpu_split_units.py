"""k_hp_split (HUFPAIR units whose lanes' streams are decoded in segments): the bits of the kernel with one half-wave per
unit, which takes the batches of more columns, for streams that fall into step, that never or hardly do (whole tables, or runs of one
code in a unit), and of very short codes; the streams that do not cost no more than that kernel's chain."""
from __future__ import annotations

import ctypes as C
import statistics

import numpy as np
import pytest
import torch

from orin_qwen_lossless_amd import _lib, synth
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
    if kind == "equal":        # sixteen pairs, equally frequent
        return ((wb & 0x807F) | (rng.integers(100, 104, wb.shape) << 7)).astype(np.uint16)
    if kind == "rare":         # 64 pairs of six bits, and one weight in two thousand of another exponent: out of step for hundreds of codes
        e = np.where(rng.random(wb.shape) < 0.0005, rng.integers(90, 92, wb.shape), rng.integers(100, 108, wb.shape))
        return ((wb & 0x807F) | (e << 7)).astype(np.uint16)
    if kind == "run":          # rows of zeros in the middle of a unit, in another two runs of one code each
        wb[rows // 2 + 1: rows // 2 + 15] = 0
        wb[2:6] = 0
        wb[9:14] = 0x3F00
    if kind == "rows":         # a row of zeros in every third unit, and one more
        wb[5::48] = 0
        wb[rows // 2 + 3] = 0
    return wb


# one unit, more than a unit per CU and more than two, the fewest and the most pair codes a lane; both orders of the chunks
@pytest.mark.parametrize("kind,units,K,R,cm", [
    ("normal", 1, 2048, 16, False), ("normal", 300, 2048, 16, True), ("normal", 513, 2048, 16, False), ("normal", 5, 4096, 16, True),
    ("normal", 257, 4096, 16, False), ("normal", 33, 1024, 16, True), ("normal", 7, 2048, 8, False), ("normal", 9, 3072, 8, True),
    ("normal", 9, 2560, 8, False), ("normal", 239, 4096, 8, False), ("normal", 257, 4096, 8, True), ("one", 3, 2048, 16, False), ("short", 3, 2048, 16, False), ("short", 2, 4096, 16, True),
    ("flat", 3, 2048, 16, False), ("flat", 2, 4096, 16, False), ("flat", 2, 2048, 8, True),
    ("equal", 1, 2048, 16, False), ("equal", 2, 4096, 4, False), ("equal", 515, 2048, 16, False), ("rare", 7, 2048, 16, True),
    ("rare", 7, 4096, 8, False), ("rare", 301, 4096, 16, False), ("rare", 33, 3072, 8, True), ("rare", 513, 2048, 16, False),
    ("run", 9, 2048, 16, False), ("run", 3, 4096, 16, False), ("run", 300, 2048, 16, True), ("run", 5, 1024, 16, False), ("run", 4, 3072, 8, False),
    ("rows", 64, 4096, 16, False), ("rows", 301, 4096, 16, True), ("rows", 500, 3072, 8, False)])
def test_split_units_have_the_bits_of_whole_ones(ops, kind, units, K, R, cm):
    rows = units * R
    wb = _matrix(kind, rows, K)
    w = enc(ops, wb, HP, R, cm, False)
    assert w.meta.format == HP and w.meta.chunk_major == cm
    xb = tbf16(synth.activations(9, K, 7))
    limit = min(8 if K <= 2048 or units <= ops.cu_count() else 6, (R * K // 64 - 128) // 48) if R * K // 64 <= 512 else 4
    for x in (xb, xb.float()):
        whole = ops.mmv(x, w)
        assert ops.last_kernel().startswith("k_huf_mmv<3, ")
        for t in {1, 2, limit}:
            y = ops.mmv(x[:t], w)
            assert ops.last_kernel().startswith("k_hp_split<")
            assert torch.equal(y, whole[:t]), t
        assert torch.equal(ops.mmv(x[:1], w, out_dtype=torch.bfloat16), whole[:1].to(torch.bfloat16))
    assert np.array_equal(bits(ops.dequant(w)), wb)
    if units > 2:                                              # a range of units that ends before the matrix, and the last one
        assert np.array_equal(bits(ops.dequant(w, R, R)), wb[R:2 * R])
        assert np.array_equal(bits(ops.dequant(w, rows - R, R)), wb[-R:])


def test_strided_and_misaligned_columns(ops):
    """Token strides of whole 16 bytes are taken; the C ABI's others, and columns that begin elsewhere, go to a half-wave per unit."""
    K, R, rows = 2048, 16, 80
    w = enc(ops, _matrix("normal", rows, K), HP, R, False, False)
    x = tbf16(synth.activations(5, K, 7))
    for xt in (x, x.float()):
        one = ops.mmv(xt, w)
        wide = torch.zeros((5, K + 24), dtype=xt.dtype, device="cuda")
        wide[:, 8: 8 + K] = xt
        assert torch.equal(ops.mmv(wide[:, 8: 8 + K], w), one) and ops.last_kernel().startswith("k_hp_split<")
        for shift, pad in ((0, 1), (1, 0), (1, 7)):
            flat = torch.zeros(shift + 5 * (K + pad), dtype=xt.dtype, device="cuda")
            view = flat[shift:].view(5, K + pad)[:, :K]
            view.copy_(xt)
            y = torch.full_like(one, 7.0)
            a = _lib.MmvArgs(view.data_ptr(), y.data_ptr(), None, view.stride(0) * view.element_size(), rows * 4, 0, 0, 0, 0, rows, 0, rows, 5, 1, 1,
                             xt.dtype == torch.bfloat16, False)
            _lib.check(_lib.lib().bf16n_mmv(C.byref(ops._cweight(w)), C.byref(a), torch.cuda.current_stream().cuda_stream, 1))
            assert ops.last_kernel().startswith("k_huf_mmv<") and torch.equal(y, one), (shift, pad)


# beyond two units per CU: rows whose planes stay in registers, rows whose planes are read again for every column, and a launch
# of three passes (columns beyond the line were slower in segments: 5120 x 4096, four 53 us, 47 by half-waves)
@pytest.mark.parametrize("K,R,most", [(2048, 16, 8), (4096, 8, 2), (3584, 8, 1), (2560, 16, 0), (3072, 16, 1)])
def test_columns_beyond_two_units_per_cu(ops, K, R, most):
    rows = (2 * ops.cu_count() + 9) * R
    wb = _matrix("normal", rows, K)
    w = enc(ops, wb, HP, R, False, False)
    x = tbf16(synth.activations(9, K, 7))
    whole = ops.mmv(x, w)
    for t in (1, 2, 3, 8):
        assert torch.equal(ops.mmv(x[:t], w), whole[:t]), t
        assert ops.last_kernel().startswith("k_hp_split<") == (t <= most), t
    assert np.array_equal(bits(ops.dequant(w)), wb)


def _us(f) -> float:
    """Median time of a call among thirty, in microseconds."""
    times = []
    f()
    for _ in range(7):
        t0, t1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        t0.record()
        for _ in range(30):
            f()
        t1.record()
        t1.synchronize()
        times.append(t0.elapsed_time(t1) * 1000 / 30)
    return statistics.median(times)


# 64 units: nine columns are nine chains side by side on an otherwise idle device, k_huf_mmv's time.  Measured here / there, us:
# rare 40 / 43 (59 with a round per segment), run 39 / 81 (136)
@pytest.mark.parametrize("kind,K", [("rare", 2048), ("run", 4096)])
def test_streams_out_of_step_take_no_longer_than_a_chain(ops, kind, K):
    w = enc(ops, _matrix(kind, 64 * 16, K), HP, 16, False, False)
    x = tbf16(synth.activations(9, K, 7))
    split = _us(lambda: ops.mmv(x[:1], w))
    assert ops.last_kernel().startswith("k_hp_split<")
    chain = _us(lambda: ops.mmv(x, w))
    assert ops.last_kernel().startswith("k_huf_mmv<")
    print(f"{kind}: {split:.1f} us, chain {chain:.1f}")
    assert split <= 1.2 * chain, (split, chain)


# The threads past the end of a run keep the places that they have found: a row of 4096 is two segments of 32, which costs two more
# rounds than normal weights (28.7 and 23.1 us), not those in which the rows behind it would fall into step again (34.6)
def test_a_row_of_zeros_leaves_the_rows_behind_it_in_step(ops):
    x = tbf16(synth.activations(1, 4096, 7))
    w, zeros = (enc(ops, _matrix(kind, 64 * 16, 4096), HP, 16, False, False) for kind in ("normal", "rows"))
    normal, rows = _us(lambda: ops.mmv(x, w)), _us(lambda: ops.mmv(x, zeros))
    assert ops.last_kernel().startswith("k_hp_split<")
    print(f"normal {normal:.1f} us, rows of zeros {rows:.1f}")
    assert rows <= 1.36 * normal, (rows, normal)
