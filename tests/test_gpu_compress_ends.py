"""The tokens at a block's end in skv_compress_append: a turn of the fold may reach
past them, and what lies there counts for nothing.
"""

from __future__ import annotations

import pytest
import torch

from test_gpu_compute import _i32

pytestmark = pytest.mark.gpu

INF = float("inf")


@pytest.mark.parametrize("m", [3, 5, 18, 33, 130])
@pytest.mark.parametrize("rows", [torch.bfloat16, torch.float32])
def test_infinite_bias(dev, m, rows) -> None:
    """A bias of +inf gives its token the whole weight, one of -inf none, also in
    the last tokens of a block (which share a turn with places that hold none)."""
    from saint_kv import ops

    g = torch.Generator().manual_seed(m)
    ch, blocks = 64, 3
    c, z = (torch.randn(1, blocks * m + 1, ch, generator=g).to(rows) for _ in range(2))
    bias = torch.randn(m, ch, generator=g)
    at = torch.randint(0, m, (ch,), generator=g)
    at[0], at[1], at[2] = 0, m - 1, 4 * ((m - 1) // 4)
    bias[at, torch.arange(ch)] = INF
    bias[(at + 1) % m, torch.arange(ch)] = -INF
    pool = torch.zeros(1, 16, ch, dtype=torch.bfloat16, device=dev)
    state = torch.zeros(1, 3, ch, device=dev)
    n = blocks * m + 1
    ops.compress_append(pool, _i32([[0]], dev), state, c.to(dev), z.to(dev), bias.to(dev), _i32([n], dev), n)
    want = c[0, : blocks * m].view(blocks, m, ch)[:, at, torch.arange(ch)].to(torch.bfloat16)
    assert torch.equal(pool[0, :blocks].cpu(), want)


@pytest.mark.parametrize("m", [4, 7, 15])
def test_state_of_a_score_that_is_minus_infinity(dev, m) -> None:
    """A token's state counts the tokens that came, one for each whose score is -inf so far."""
    from saint_kv import ops

    ch = 8
    for n in range(1, m):
        z = torch.full((1, n, ch), -INF, dtype=torch.bfloat16, device=dev)
        c = torch.ones(1, n, ch, dtype=torch.bfloat16, device=dev)
        pool, state = torch.zeros(1, 16, ch, dtype=torch.bfloat16, device=dev), torch.zeros(1, 3, ch, device=dev)
        ops.compress_append(pool, _i32([[0]], dev), state, c, z, torch.zeros(m, ch, device=dev), _i32([n], dev), n)
        assert state[0, :, 0].tolist() == [-INF, n, n] and bool((state[0] == state[0, :, :1]).all())
