"""skv_compress_append at the edges of its work split: blocks of 1 to 128
tokens around the slice counts (1, 4 and 16 lane groups per entry), channel
counts that leave a 128-channel block partly empty, and blocks that end,
begin and continue inside one call.  Same oracle and bound as
test_gpu_compute.py.
"""

from __future__ import annotations

import pytest
import torch

from oracle import reference_cpu as ref
from test_gpu_compute import _compress_case, _i32

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,channels", [(1, 8), (2, 2048), (4, 136), (5, 64), (31, 128), (32, 576), (33, 264), (128, 8)])
def test_compress_slices(dev, m, channels) -> None:
    # ragged chunks: nothing new, one token, up to a block's end, past several
    # blocks, a call that both completes and leaves blocks behind
    chunks = [[0, 1, m, 3 * m + 1], [1, m, m - 1, 17 * m], [m, 0, 2 * m + 3, 1], [1, 1, 1, m]]
    _compress_case(dev, batch=4, m=m, channels=channels, chunks=chunks, fp8=False, seed=m + channels)


@pytest.mark.parametrize("m", [4, 8, 32])
def test_compress_infinite_scores(dev, m) -> None:
    """A token whose score is -inf has no weight wherever it stands; a channel
    whose scores are all -inf, or hold a NaN, pools to NaN (softmax's values)."""
    from saint_kv import ops

    g = torch.Generator().manual_seed(m)
    ch = 16
    c = torch.randn(1, 2 * m, ch, generator=g).to(torch.bfloat16)
    z = torch.randn(1, 2 * m, ch, generator=g).to(torch.bfloat16)
    inf = float("inf")
    z[0, 0, 0] = z[0, m - 1, 1] = z[0, 1:m, 2] = -inf  # first, last, all but the first token
    z[0, m: 2 * m, 3] = -inf                           # a whole block
    z[0, m // 2, 4] = float("nan")
    bias = torch.randn(m, ch, generator=g)
    pool = torch.zeros(1, 16, ch, dtype=torch.bfloat16, device=dev)
    state = torch.zeros(1, 3, ch, device=dev)
    ops.compress_append(pool, _i32([[0]], dev), state, c.to(dev), z.to(dev), bias.to(dev), _i32([2 * m], dev), 2 * m)
    want = ref.compress_pool(c.view(2, m, ch), z.view(2, m, ch), bias)
    bound = ref.pooling_bound(c.view(2, m, ch), z.view(2, m, ch), bias)
    got = pool[0, :2].float().cpu()
    assert torch.equal(torch.isnan(got), torch.isnan(want))
    live = ~torch.isnan(want)
    assert bool(((got - want).abs() <= bound)[live].all())
    assert bool(torch.isnan(got[1, 3])) and bool(torch.isnan(got[0, 4]))
