"""An entry's bits do not depend on how its tokens came: a prompt at once, in
chunks of several lengths, a token at a time, or in decode steps; for every
block length, entry format and row type.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from test_gpu_compute import _i32

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,ch,entry,rows", [
    (1, 8, "bf16", torch.bfloat16), (15, 136, "bf16", torch.bfloat16), (16, 576, "fp8", torch.bfloat16),
    (17, 64, "f32", torch.float32), (31, 576, "fp8", torch.float32), (32, 576, "fp8", torch.bfloat16),
    (64, 2048, "bf16", torch.bfloat16), (100, 264, "bf16", torch.float32), (128, 576, "fp8", torch.bfloat16),
    (130, 8, "f32", torch.float32),
])
def test_bits_do_not_depend_on_the_calls(dev, m, ch, entry, rows) -> None:
    from saint_kv import ops
    from saint_kv._lib import fp8_entry_bytes

    g = torch.Generator().manual_seed(m)
    b, t = 2, 3 * m + m // 2
    c, z = (torch.randn(b, t, ch, generator=g).to(dev, rows) for _ in range(2))
    bias = torch.randn(m, ch, generator=g).to(dev)
    dtype = {"bf16": torch.bfloat16, "f32": torch.float32, "fp8": torch.uint8}[entry]
    got = []
    for step in (t, 1, 7, m + 3, 2 * m):
        pool = torch.zeros(b, 16, fp8_entry_bytes(ch) if entry == "fp8" else ch, device=dev, dtype=dtype)
        state = torch.zeros(b, 3, ch, device=dev)
        for lo in range(0, t, step):
            hi = min(lo + step, t)
            ops.compress_append(pool, _i32([[0], [1]], dev), state, c[:, lo:hi].contiguous(), z[:, lo:hi].contiguous(),
                                bias, _i32([hi] * b, dev), hi - lo)
        got.append((step, pool, state))
    for step, pool, state in got[1:]:
        assert torch.equal(pool.view(torch.uint8), got[0][1].view(torch.uint8)), step
        assert t % m == 0 or torch.equal(state, got[0][2]), step


@pytest.mark.parametrize("m,fp8", [(32, True), (128, False), (128, True)])
def test_decode_steps_give_the_prompt_bits(dev, m, fp8) -> None:
    from saint_kv.decode import DecodeCache, LayerSpec

    lens0 = np.array([m - 3, 2 * m, m // 2])
    steps, b = m, 3
    t = int(lens0.max()) + steps
    g = torch.Generator().manual_seed(m)
    rows = {k: torch.randn(b, t, 576, generator=g).to(dev, torch.bfloat16) for k in ("kv", "c", "z")}
    bias = torch.randn(m, 576, generator=g).to(dev)
    caches = []
    for lens in (lens0, lens0 + steps):
        cache = DecodeCache([LayerSpec("hca", m=m, fp8=fp8)], b, t + 1, block_size=16, window=8, device=dev)
        cache.bias[0].copy_(bias)
        cache.prefill(lens, data=[rows])
        caches.append(cache)
    at = torch.arange(b, device=dev)
    for s in range(steps):
        for k, v in rows.items():
            caches[0].inputs[0][k].copy_(v[at, torch.as_tensor(lens0 + s, device=dev)])
        caches[0].step()
    caches[0].check_status()
    for q in range(b):
        n = int(lens0[q] + steps)
        for e in range(n // m):
            x, y = (h.pool[0][int(h.groups[0].block_table[q, 0]), e] for h in caches)
            assert torch.equal(x, y), (q, e)
        if n % m:
            assert torch.equal(caches[0].state[0][q], caches[1].state[0][q]), q


@pytest.mark.parametrize("m,t,ch,rows", [(4, 1, 576, torch.bfloat16), (4, 3, 2048, torch.bfloat16),
                                         (128, 1, 136, torch.float32), (32, 6, 576, torch.float32),
                                         (16, 40, 264, torch.bfloat16)])
def test_many_sequences_at_once(dev, m, t, ch, rows) -> None:
    """Workgroups shared by several blocks of channels give the bits of calls of a few sequences."""
    from saint_kv import ops

    g = torch.Generator().manual_seed(m + t)
    b, part, had = 513, 3, 2  # the blocks hold two tokens before the call
    c, z = (torch.randn(b, had + t, ch, generator=g).to(dev, rows) for _ in range(2))
    bias = torch.randn(m, ch, generator=g).to(dev)
    new = torch.randint(0, t + 1, (b,), generator=g, dtype=torch.int32).to(dev)
    got = []
    for size in (b, part):
        pool = torch.zeros(b, 16, ch, dtype=torch.bfloat16, device=dev)
        state = torch.zeros(b, 3, ch, device=dev)
        for lo in range(0, b, size):
            at = slice(lo, min(lo + size, b))
            bt = _i32([[i] for i in range(lo, at.stop)], dev)
            n = new[at]
            ops.compress_append(pool, bt, state[at], c[at, :had], z[at, :had], bias, torch.full_like(n, had), had)
            ops.compress_append(pool, bt, state[at], c[at, had:], z[at, had:], bias, n + had, n)
        got.append((pool, state))
    assert torch.equal(got[0][0], got[1][0])
    live = (had + new) % m > 0  # a state is left
    assert torch.equal(got[0][1][live], got[1][1][live]) and bool(live.any())
