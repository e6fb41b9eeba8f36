"""reset() of the drop-in layers recorded in a graph: it makes nothing of its own,
so that an eager reset before the first replay, and one on another stream, give
every page back.
"""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch", [1, 3, 4, 9])
def test_first_reset_in_a_graph(dev, batch) -> None:
    from saint_kv.kv_cache import SWAKVCacheLayer

    g = torch.Generator(device=dev).manual_seed(batch)
    layer = SWAKVCacheLayer(64, 32, batch_size=batch, device=dev, dtype=torch.float32, block_size=16)
    rows = layer._rows
    k, v = (torch.randn(batch, 40, 32, generator=g, device=dev) for _ in range(2))

    def held() -> tuple:
        torch.cuda.synchronize()
        return int(rows.free_top.item()), rows.lens.tolist()

    def fill() -> None:
        got = layer.append(k, v)
        assert torch.equal(got[0], k) and torch.equal(got[1], v)
        assert held() == (rows.pool.shape[0] - 3 * batch, [40] * batch)

    empty = (rows.pool.shape[0], [0] * batch)
    fill()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        layer.reset()
    rows.length = 40  # recorded, not run
    before = torch.cuda.memory_allocated()
    layer.reset()
    assert torch.cuda.memory_allocated() == before
    assert held() == empty
    for _ in range(3):
        fill()
        graph.replay()
        rows.length = 0
        assert held() == empty
    fill()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        layer.reset()
    torch.cuda.current_stream().wait_stream(side)
    assert held() == empty
