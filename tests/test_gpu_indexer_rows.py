"""skv_indexer_scores for several query tokens per sequence: the scores of
every token are the bits that a call for that token alone gives (which
test_gpu_compute.py holds to the fp64 oracle), at the edges of the kernel's
tiles: 8 tokens and 128 entries per workgroup, runs of several tiles, heads
and channels that fill no whole block, and unmapped pages.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("t,h,c,n_max", [
    (6, 64, 128, 129), (8, 1, 8, 127), (9, 16, 32, 128), (17, 17, 40, 300), (33, 33, 64, 1000), (64, 64, 128, 2500),
    (7, 64, 120, 1),
])
def test_indexer_scores_rows(dev, t, h, c, n_max) -> None:
    from saint_kv import ops

    g = torch.Generator().manual_seed(t * 100 + h)
    batch, bs = 3, 16
    n_ent = torch.tensor([n_max, n_max // 2, 0], dtype=torch.int32, device=dev)
    pages = -(-n_max // bs)
    table = np.random.default_rng(t).permutation(batch * pages).reshape(batch, pages).astype(np.int32)
    table[0, pages // 2] = -1  # unmapped: scores -inf
    table = torch.as_tensor(table, device=dev)
    pool = torch.randn(batch * pages, bs, c, generator=g).to(torch.bfloat16).to(dev)
    q = torch.randn(batch, t, h, c, generator=g).to(torch.bfloat16).to(dev)
    q[0, 1, 0, 0] = float("inf")  # NaN and infinite products follow the same rule
    w = torch.randn(batch, t, h, generator=g).to(dev)
    got = torch.full((batch, t, n_max + 3), 7.0, device=dev)
    ops.indexer_scores(q, w, pool, table, n_ent, got, max_entries=n_max)
    for i in range(t):
        one = torch.full((batch, 1, n_max + 3), 7.0, device=dev)
        ops.indexer_scores(q[:, i:i + 1].contiguous(), w[:, i:i + 1].contiguous(), pool, table, n_ent, one,
                           max_entries=n_max)
        assert torch.equal(got[:, i].view(torch.int32), one[:, 0].view(torch.int32)), i


@pytest.mark.parametrize("batch,t,h,c,n_max", [(120, 6, 64, 128, 129), (100, 7, 64, 120, 1), (8, 33, 33, 64, 1000),
                                               (64, 9, 50, 40, 513), (20, 6, 32, 128, 127), (12, 17, 17, 72, 300)])
def test_large_queries_of_many_sequences(dev, batch, t, h, c, n_max) -> None:
    """Queries that take the rows' kernel only where its tiles fill the device, against a token at a time."""
    from saint_kv import ops

    g = torch.Generator().manual_seed(batch + h)
    n_ent = torch.randint(0, n_max + 1, (batch,), generator=g, dtype=torch.int32)
    n_ent[0], n_ent[-1] = n_max, 0
    n_ent = n_ent.to(dev)
    pages = -(-n_max // 16)
    table = torch.randperm(batch * pages, generator=g).view(batch, pages).to(torch.int32).to(dev)
    pool = torch.randn(batch * pages, 16, c, generator=g).to(torch.bfloat16).to(dev)
    q = torch.randn(batch, t, h, c, generator=g).to(torch.bfloat16).to(dev)
    w = torch.randn(batch, t, h, generator=g).to(dev)
    got = torch.full((batch, t, n_max), 7.0, device=dev)
    ops.indexer_scores(q, w, pool, table, n_ent, got)
    for i in range(t):
        one = torch.full((batch, 1, n_max), 7.0, device=dev)
        ops.indexer_scores(q[:, i:i + 1].contiguous(), w[:, i:i + 1].contiguous(), pool, table, n_ent, one)
        assert torch.equal(got[:, i].view(torch.int32), one[:, 0].view(torch.int32)), i
