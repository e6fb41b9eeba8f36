"""Calls of skv_compress_append whose rows would need more workgroups than a
launch can have (2^32 work items): each workgroup takes several turns.  The
rows are views of one row, so that the calls hold next to no memory.
"""

from __future__ import annotations

import pytest
import torch

from test_gpu_compute import _i32

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_streams,in_len", [(1, 1 << 28), (16, 1 << 25), (3, (1 << 27) + 5)])
def test_more_blocks_than_a_launch_holds(dev, n_streams, in_len) -> None:
    from saint_kv import ops

    g = torch.Generator().manual_seed(n_streams)
    n, m, ch = 40, 1, 8
    streams = []
    for _ in range(n_streams):
        c, z = (torch.randn(1, 1, ch, generator=g).to(dev, torch.bfloat16).expand(1, in_len, ch) for _ in range(2))
        streams.append((torch.zeros(3, 16, ch, dtype=torch.bfloat16, device=dev), _i32([[2, 0, 1]], dev),
                        torch.zeros(1, 3, ch, device=dev), c, z, torch.randn(m, ch, generator=g).to(dev)))
    ops.compress_append_streams(streams, _i32([n], dev), n)
    for pool, bt, _, c, _, _ in streams:
        assert torch.equal(pool[bt[0].long()].view(-1, ch)[:n], c[0, :n])
        assert not pool[bt[0].long()].view(-1, ch)[n:].any()
