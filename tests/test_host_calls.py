"""The dense product's native call (csrc/host_calls.cpp): it takes the plain case with the result of the Python layer's, and
answers everything else with None, so that the Python layer's checks and messages hold."""
from __future__ import annotations

import sys
import types
import warnings

import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

from orin_qwen_lossless_amd import build, ops, synth


class Sub(torch.Tensor):
    pass


class Pass(TorchDispatchMode):
    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


def _calls():
    return ops._host_calls or ops._host()


def test_nothing_on_the_host_is_taken():
    meta = ops.Meta(1, 512, 4, 1, False, False, 256, 512, 640, 700)
    w = ops.Weight(torch.zeros(4 * 512, dtype=torch.uint8), torch.zeros(1024, dtype=torch.uint8), meta)
    x = torch.zeros(1, 512, dtype=torch.bfloat16)
    for args in ((x, w, True, True), (x, None, True, True), (None, w, True, True), (x, w)):
        assert _calls().mmv(*args) is None
    for args in ((x, w, 8, 1 << 20), (x, w)):
        assert _calls().linear(*args) is None
    with pytest.raises(ValueError, match="device"):
        ops.mmv(x, w)


def test_without_the_extension_module_calls_go_the_general_way(monkeypatch):
    monkeypatch.setattr(ops, "_host_calls", None)
    monkeypatch.setitem(sys.modules, "orin_qwen_lossless_amd._host", None)  # an import that fails
    meta = ops.Meta(1, 512, 4, 1, False, False, 256, 512, 640, 700)
    w = ops.Weight(torch.zeros(4 * 512, dtype=torch.uint8), torch.zeros(1024, dtype=torch.uint8), meta)
    x = torch.zeros(1, 512, dtype=torch.bfloat16)
    with pytest.warns(RuntimeWarning, match="build it with"), pytest.raises(ValueError, match="device"):
        ops.mmv(x, w)
    for call in (ops.mmv, ops.linear):                   # (said once)
        with warnings.catch_warnings(), pytest.raises(ValueError, match="device"):
            warnings.simplefilter("error")
            call(x, w)


def test_a_module_built_for_another_torch_is_not_used_and_is_built_again(monkeypatch):
    assert _calls().built_for == build.torch_release()
    stale = types.ModuleType("_host")
    stale.built_for = "1.0 0"
    stale.bind = stale.mmv = stale.linear = lambda *_: pytest.fail("called")
    monkeypatch.setattr(ops, "_host_calls", None)
    for module in (stale, types.SimpleNamespace(bind=stale.bind)):  # (before there was a release in it)
        monkeypatch.setitem(sys.modules, "orin_qwen_lossless_amd._host", module)
        ops._host_calls = None
        with pytest.warns(RuntimeWarning, match="another release of torch"):
            assert ops._host().mmv(None, None, True, True) is None
    started = []
    monkeypatch.setattr(build.subprocess, "run", lambda cmd, **_: started.append(cmd) or types.SimpleNamespace(returncode=1, stdout="", stderr=""))
    build._build_host(False)
    assert not started                                   # up to date
    monkeypatch.setattr(build, "torch_release", lambda: "1.0 0")
    with pytest.raises(RuntimeError, match="building"):
        build._build_host(False)
    assert started


@pytest.mark.gpu
def test_the_plain_product_and_nothing_else(ops):
    rows, K = 200, 1024
    src = torch.from_numpy(synth.weights(rows, K, 3).view("int16")).view(torch.bfloat16)
    fmt, R, cm, fo, w64 = ops.choose(rows, K)
    plane, aux, meta = ops.encode(src, fmt, R, cm, fo, w64)
    w = ops.upload(plane, aux, meta, "cuda")
    x = synth.weights_torch(9, K, 5, "cuda")
    for xt in (x, x.float()):
        for t in (1, 2, 9):
            for out_bf16 in (False, True):
                for multi in (False, True):
                    y = _calls().mmv(xt[:t], w, out_bf16, multi)
                    ref = ops._mmv_common(xt[:t], w, None, 0, out_bf16, False, multi)
                    assert y.dtype == ref.dtype and y.shape == ref.shape and torch.equal(y, ref)
    wide = torch.zeros(9, K + 8, dtype=torch.bfloat16, device="cuda")
    wide[:, :K] = x
    assert torch.equal(_calls().mmv(wide[:, :K], w, True, True), _calls().mmv(x, w, True, True))
    short = ops.Weight(w.plane[:-K], w.aux, meta)
    moved = ops.Weight(torch.cat([w.plane, w.plane])[1: rows * K + 1], w.aux, meta)
    for bad in (x[:, :-8], x[:, ::2], x.half(), x[0], x[:0], x[None], x.cpu(), torch.cat([x, x], 1)[:, 1: K + 1], x.to_sparse(),
                x.as_subclass(Sub), wide[:, 1: K + 1]):
        assert _calls().mmv(bad, w, True, True) is None and _calls().linear(bad, w, 8, 1 << 26) is None
    assert _calls().mmv(x.float(), w, True, True) is not None and _calls().linear(x.float(), w, 8, 1 << 26) is None
    # numbers that are none, or none of these (an error that was left set would come up in the call after it)
    for gemv_tokens, chunk_bytes in (("n", 1 << 26), (8, None), (-1, 1 << 26), (8, -1), (1 << 70, 1 << 26), (8, 1 << 70), (8.5, 1 << 26)):
        assert _calls().linear(x, w, gemv_tokens, chunk_bytes) is None
        assert torch.equal(_calls().linear(x, w, 8, 1 << 26), ops.linear(x, w))
    assert _calls().mmv(x, w, True) is None and _calls().linear(x, w, 8) is None
    for refused in (short, moved):
        assert _calls().mmv(x, refused, True, True) is None and _calls().linear(x, refused, 8, 1 << 26) is None
    with Pass():
        assert _calls().mmv(x, w, True, True) is None and _calls().linear(x, w, 8, 1 << 26) is None
    seen = []
    torch.vmap(lambda v: seen.extend([_calls().mmv(v, w, True, True), _calls().linear(v, w, 8, 1 << 26)]) or v)(x[None])
    assert seen == [None, None]
    assert not _calls().mmv(torch.nn.Parameter(x.float()), w, False, True).requires_grad
    # linear: GEMV columns, columns up to the matrix's own number of them, decoded in one piece (a graph of x's gradient with
    # it) and, beyond a piece, not at all
    most = ops.gemv_max_tokens(w)
    big = synth.weights_torch(most + 1, K, 6, "cuda")
    for t in (1, 8, 9, most):
        assert torch.equal(_calls().linear(big[:t], w, 8, 1 << 26), ops._mmv_common(big[:t], w, None, 0, True, False)), t
    y = _calls().linear(big, w, 8, rows * K * 2)
    assert torch.equal(y, torch.nn.functional.linear(big, ops.dequant(w)))
    assert _calls().linear(big, w, 8, rows * K * 2 - 1) is None
    leaf = big.clone().requires_grad_()
    ops.linear(leaf, w).sum().backward()
    assert torch.equal(leaf.grad, torch.ones_like(y) @ ops.dequant(w))
    # the C ABI's refusals come back as its status
    fo_meta = ops.Meta(*meta.__dict__.values())
    object.__setattr__(fo_meta, "frag_order", True)
    with pytest.raises(ValueError, match="fragment-order"):
        ops.mmv(x, ops.Weight(w.plane, w.aux, fo_meta))
