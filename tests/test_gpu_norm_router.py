"""bf16n_add_rmsnorm_mmv (the router GEMV that forms its own input): bit for bit what the two launches it stands for give."""
from __future__ import annotations

import pytest
import torch

from orin_qwen_lossless_amd import synth
from test_gpu_kernels import NIB, enc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 255, 256])
@pytest.mark.parametrize("T,addends,gamma", [(1, 1, False), (3, 2, True), (16, 3, False)])
def test_router_that_forms_its_own_input(ops, rows, T, addends, gamma):
    g = torch.Generator(device="cuda").manual_seed(rows + T)
    wb = synth.weights(rows, 2048, rows)
    wb[:, 7::97] = 0x4500  # escaped weights
    w = enc(ops, wb, NIB, 0, False, False)
    xs = [torch.randn((T, 2048), generator=g, device="cuda").to(torch.bfloat16) for _ in range(addends)] + [None] * (3 - addends)
    gm = torch.randn(2048, generator=g, device="cuda").to(torch.bfloat16) if gamma else None
    y, s, p = ops.add_rmsnorm_mmv(xs[0], w, xs[1], xs[2], gamma=gm)
    assert ops.last_kernel() == "k_norm_nib_mmv"
    y2, s2 = ops.add_rmsnorm(xs[0], xs[1], xs[2], gamma=gm, want_sum=True)
    assert torch.equal(y, y2) and torch.equal(s, s2)
    assert torch.equal(p, ops.mmv(y2, w, multi_col=False))


def test_router_that_forms_its_own_input_refuses_other_shapes(ops):
    x = torch.zeros((1, 1024), dtype=torch.bfloat16, device="cuda")
    w = enc(ops, synth.weights(16, 1024, 1), NIB, 0, False, False)
    with pytest.raises(ValueError):
        ops.add_rmsnorm_mmv(x, w)


def test_router_that_forms_its_own_input_refuses_results_that_overlap(ops):
    """Every block reads the token's inputs while others write: a result over an input or over another result is refused on
    the host; results that touch end to end are not."""
    import ctypes as C

    from orin_qwen_lossless_amd import _lib

    T, n, rows, y_tok = 3, 2048, 32, 40
    row, prod = T * n * 2, (2 * y_tok + rows) * 4  # bytes
    w = enc(ops, synth.weights(rows, n, 4), NIB, 0, False, False)
    cw = ops._cweight(w)
    buf = synth.activations_torch(1, 8 * T * n, 5, "cuda").view(torch.uint8).view(-1)
    base = buf.data_ptr()
    assert base % 16 == 0 and prod < row
    at = {k: base + i * row for i, k in enumerate(("a", "b", "c", "gamma", "y_sum", "y_norm", "y"))}

    def call(**moved):
        p = dict(at, **moved)
        return _lib.lib().bf16n_add_rmsnorm_mmv(p["a"], p["b"], p["c"], p["gamma"], p["y_sum"], p["y_norm"], T, n, C.c_float(1e-6), C.byref(cw),
                                                p["y"], y_tok, ops._stream())

    assert call() == 0
    assert call(y=at["y_norm"] - prod, y_sum=at["y"]) == 0  # y ends where y_norm begins
    torch.cuda.synchronize()
    for k in ("a", "b", "c", "y_sum", "y_norm"):
        assert call(y=at[k]) != 0 and call(y=at[k] + row - 4) != 0 and call(y=at[k] - prod + 4) != 0, k
    assert call(y=at["gamma"] + 2 * n - 4) != 0 and call(y_sum=at["gamma"]) != 0
    assert call(y_sum=at["y_norm"]) != 0 and call(y_norm=at["y_sum"] + row - 16) != 0
    for k in ("a", "b", "c"):
        assert call(y_norm=at[k]) != 0 and call(y_sum=at[k] + 16) != 0, k
    torch.cuda.synchronize()
