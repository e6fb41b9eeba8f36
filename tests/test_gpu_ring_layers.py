"""skv_ring_append_layers: rings of one batch in one launch hold the rows that a
call per ring writes, for rings of other windows, row sizes and source strides,
past the rings that one launch takes.
"""

from __future__ import annotations

import pytest
import torch

from test_gpu_compute import _i32

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_rings", [1, 3, 16, 17])
def test_ring_layers_equal_single_calls(dev, n_rings) -> None:
    from saint_kv import ops

    g = torch.Generator().manual_seed(n_rings)
    b, t, lens, new = 3, 150, [150, 40, 7], [150, 3, 0]
    rings, want = [], []
    for i in range(n_rings):
        window, ch = [128, 1, 17, 33][i % 4], [576, 8, 136][i % 3]
        src = torch.randn(b, t, 2, ch, generator=g).to(dev, torch.bfloat16)[:, :, i % 2]  # rows with a gap where i % 2
        ring = torch.zeros(b, window, ch, dtype=torch.bfloat16, device=dev)
        rings.append((ring, src))
        want.append(ring.clone())
        ops.ring_append(want[-1], _i32(lens, dev), src, _i32(new, dev))
        # by hand: the newest rows of each sequence, slot = position % window
        for s in range(b):
            for pos in range(max(lens[s] - new[s], lens[s] - window), lens[s]):
                assert torch.equal(want[-1][s, pos % window], src[s, pos - (lens[s] - new[s])])
    ops.ring_append_layers(rings, _i32(lens, dev), _i32(new, dev))
    for (ring, _), w in zip(rings, want):
        assert torch.equal(ring, w)
    ops.ring_append_layers([], _i32(lens, dev), 1)
