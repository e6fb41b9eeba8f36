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


@pytest.mark.parametrize("m,fp8", [(4, True), (4, False), (8, True), (15, False)])
def test_short_blocks_are_the_same_at_once_and_by_tokens(dev, m, fp8) -> None:
    """Entries (their fp8 codes) and states of blocks of one slice do not depend
    on how the tokens were split over calls."""
    from saint_kv import ops
    from saint_kv._lib import fp8_entry_bytes

    g = torch.Generator().manual_seed(m)
    b, t, ch = 2, 40 * m + m // 2, 576
    c, z = (torch.randn(b, t, ch, generator=g).to(dev, torch.bfloat16) for _ in range(2))
    bias = torch.randn(m, ch, generator=g).to(dev)
    got = []
    for step in (t, 1, m + 3):
        pool = torch.zeros(b, 64, fp8_entry_bytes(ch) if fp8 else ch, device=dev,
                           dtype=torch.uint8 if fp8 else torch.bfloat16)
        state = torch.zeros(b, 3, ch, device=dev)
        for lo in range(0, t, step):
            hi = min(lo + step, t)
            ops.compress_append(pool, _i32([[0], [1]], dev), state, c[:, lo:hi].contiguous(), z[:, lo:hi].contiguous(),
                                bias, _i32([hi] * b, dev), hi - lo)
        got.append((pool, state))
    for pool, state in got[1:]:
        assert torch.equal(pool.view(torch.uint8), got[0][0].view(torch.uint8)) and torch.equal(state, got[0][1])
