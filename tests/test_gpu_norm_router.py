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
    y2, s2 = ops.add_rmsnorm(xs[0], xs[1], xs[2], gamma=gm, want_sum=True)
    assert torch.equal(y, y2) and torch.equal(s, s2)
    assert torch.equal(p, ops.mmv(y2, w, multi_col=False))


def test_router_that_forms_its_own_input_refuses_other_shapes(ops):
    x = torch.zeros((1, 1024), dtype=torch.bfloat16, device="cuda")
    w = enc(ops, synth.weights(16, 1024, 1), NIB, 0, False, False)
    with pytest.raises(ValueError):
        ops.add_rmsnorm_mmv(x, w)
