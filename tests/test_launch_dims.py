"""Launch shapes and rules that need no GPU: no CU gets more wavefronts than an even split gives (csrc/launch_dims.h); the
router's launch forms its own input where that was measured to be the faster way."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.skipif(shutil.which("g++") is None, reason="no g++")
def test_wavefronts_are_spread_over_the_device(tmp_path):
    exe = str(tmp_path / "launch_dims")
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-fsanitize=undefined", "-fno-sanitize-recover=undefined",
                    "-I" + os.path.join(ROOT, "orin_qwen_lossless_amd", "csrc"), os.path.join(ROOT, "tests", "cpp", "launch_dims.cpp"), "-o", exe],
                   check=True, capture_output=True, timeout=120)
    out = subprocess.run([exe], check=True, capture_output=True, text=True, timeout=60).stdout.splitlines()
    for ln, (cus, full) in zip(out, [(c, f) for c in (256, 64, 1) for f in (8, 16)]):
        head, values = ln.split(": ")
        over, largest, filled = map(int, values.split())
        assert head == f"{cus} {full}" and over == 0 and largest <= 16 and filled == full, ln
    assert out[-1] == "9 9 8"


@pytest.mark.parametrize("rows,last", [(64, 64), (256, 16), (512, 8), (1024, 4), (2048, 2), (4096, 1), (8192, 0)])
def test_where_the_router_forms_its_own_input(rows, last):
    """Last token count at which one launch was the faster way, by matrix rows."""
    import torch

    from orin_qwen_lossless_amd import decode_step, ops

    buf = torch.empty(16, dtype=torch.uint8)
    w = ops.Weight(buf, buf, ops.Meta(ops.FMT_NIBBLE, 2048, rows, 0, False, False, 256, 256, 256, 256))
    assert [T for T in range(130) if ops.add_rmsnorm_mmv_supported(w, T)] == list(range(1, last + 1))
    x = torch.empty(17, dtype=torch.bfloat16)
    assert not last or ops.add_rmsnorm_mmv_supported(w, 1, x[:16], x[:8]) and not ops.add_rmsnorm_mmv_supported(w, 1, x[:16], x[1:])
    if rows == decode_step.E:  # what a step reports is what it launches
        per_layer = [decode_step.launches_per_layer(ops, T, False) for T in (12, 13, 16, 17)]
        assert per_layer == [7, 8, 8, 9]


@pytest.mark.parametrize("n_experts,k,n_slots,last", [(256, 8, 9, 12), (64, 2, 10, 12), (256, 8, 8, 8), (257, 8, 9, 8), (512, 8, 9, 8),
                                                      (256, 10, 11, 8), (64, 4, 4, 8), (256, 9, 9, 12), (256, 1, 25, 8)])
def test_where_selection_and_lists_are_one_launch(n_experts, k, n_slots, last):
    """Nine to twelve tokens only where one launch was measured to be ahead."""
    from orin_qwen_lossless_amd import ops

    assert ops.topk_route_one_launch_tokens(n_experts, k, n_slots) == last
