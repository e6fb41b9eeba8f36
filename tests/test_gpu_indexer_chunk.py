"""``indexer_topk`` reading its keys in place, its causal mask worked out in the kernels.

Against the general route (``lightning_indexer_scores``, then ``ops.topk_select``
with each row's visible count): both give the same score bits, so the picks are
equal.  The sizes cross the line between the two score kernels (6 tokens), tiles
that no token of a group sees, token groups that straddle the first visible
entry, entries past those in use, and keys that have to be copied first.
"""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("b,t_new,h,c,offset,n_blocks,rows,m,top_k,form", [
    (1, 1, 4, 32, 16, 4, 4, 4, 16, "plain"),  # fewer entries than picks
    (2, 5, 8, 64, 1019, 256, 300, 4, 64, "plain"),  # the last count before the grouped kernel, spare entries
    (3, 6, 16, 128, 0, 70, 70, 4, 512, "plain"),  # most tokens see nothing
    (2, 9, 64, 128, 2047, 514, 520, 4, 512, "plain"),  # a group of one token
    (1, 300, 33, 24, 100, 400, 400, 1, 100, "plain"),  # whole tiles unseen by the first groups
    (2, 17, 4, 8, 500, 129, 140, 4, 40, "strided"),
    (2, 17, 4, 8, 500, 129, 140, 4, 40, "f32"),
    (1, 7, 4, 8, 40, 30, 30, 2 ** 40, 5, "plain"),  # a block longer than any position
    (1, 2, 64, 128, 65536, 16384, 16384, 4, 1024, "plain"),  # the last size of this route
    (1, 2, 64, 128, 65540, 16385, 16400, 4, 1024, "plain"),  # the first past it
])
def test_picks_equal_the_general_route(b, t_new, h, c, offset, n_blocks, rows, m, top_k, form) -> None:
    from saint_kv import ops
    from saint_kv.indexer import indexer_topk, lightning_indexer_scores

    dev = torch.device("cuda:0")
    g = torch.Generator().manual_seed(t_new * 7 + c)
    q = torch.randn(b, t_new, h, c, generator=g).to(dev, torch.bfloat16)
    w = torch.randn(b, t_new, h, generator=g).to(dev)
    k = torch.randn(b, rows, c, generator=g).to(dev, torch.float32 if form == "f32" else torch.bfloat16)
    if form == "strided":
        k = k.transpose(0, 1).contiguous().transpose(0, 1)
    got = indexer_topk(q, w, k, cache_offset=offset, total_len=offset + t_new, n_blocks=n_blocks, m=m, top_k=top_k)
    k_eff = min(top_k, n_blocks)
    scores = lightning_indexer_scores(q, k[:, :n_blocks], w).view(b * t_new, n_blocks)
    seen = [min((offset + t) // m, n_blocks) for t in range(t_new)] * b
    want = torch.empty(b * t_new, k_eff, dtype=torch.int32, device=dev)
    ops.topk_select(scores, torch.tensor(seen, dtype=torch.int32, device=dev), n_blocks, k_eff, want)
    assert got.dtype == torch.int64 and tuple(got.shape) == (b, t_new, k_eff)
    assert torch.equal(got.view(b * t_new, k_eff), want.long())


@pytest.mark.parametrize("m,seen", [(2 ** 40, 0), (2 ** 31 - 1, 0), (2 ** 31 - 2, 1)])
def test_last_position(m, seen) -> None:
    """The position 2^31 - 2 and blocks about as long: an entry is seen once its block is complete before it."""
    from saint_kv.indexer import indexer_topk

    dev, last = torch.device("cuda:0"), 2 ** 31 - 2
    q, k = torch.ones(1, 1, 4, 8, device=dev), torch.ones(1, 3, 8, device=dev)
    got = indexer_topk(q, torch.ones(1, 1, 4, device=dev), k, cache_offset=last, total_len=last + 1, n_blocks=3, m=m, top_k=2)
    assert got.tolist() == [[[0, -1] if seen else [-1, -1]]]
