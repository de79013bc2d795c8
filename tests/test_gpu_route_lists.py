"""k_route: the expert-sorted lists against a stable sort, for the counts of ids with vector loads and others, rows that are
and are not aligned for them, and token counts at the ends of a round and of a chunk of rounds."""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_used", [1, 2, 3, 4, 6, 8, 9])
@pytest.mark.parametrize("tokens", [1, 63, 1025, 65536, 65537])
def test_lists_are_a_stable_sort(ops, n_used, tokens):
    E = 20
    g = torch.Generator().manual_seed(n_used + tokens)
    ids = torch.rand((tokens, E), generator=g).argsort(1)[:, :n_used].to(torch.int32)
    order = torch.sort(ids.reshape(-1), stable=True)
    counts = torch.bincount(ids.reshape(-1).long(), minlength=E)
    bounds = torch.cat([torch.zeros(1, dtype=torch.long), counts.cumsum(0)]).to(torch.int32)
    dst = order.indices.to(torch.int32)
    for pad, shift in ((0, 0), (1, 0), (2, 1), (8, 2)):     # row strides and starts of every alignment
        flat = torch.zeros(tokens * (n_used + pad) + 8, dtype=torch.int32, device="cuda")
        view = flat[shift: shift + tokens * (n_used + pad)].view(tokens, n_used + pad)[:, :n_used]
        view.copy_(ids)
        for given in (view, view.long()) if pad == 0 else (view,):
            for per_slot in (False, True):
                s, d, b = (t.cpu() for t in ops.mm_ids_route(given, E, per_slot))
                assert torch.equal(b, bounds) and torch.equal(d, dst)
                assert torch.equal(s, dst if per_slot else dst // n_used)
