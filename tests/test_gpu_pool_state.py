"""The pooling state that appends and decode steps share: a block gives one
entry, whichever of them brought its tokens, also where scores are infinite or
NaN.  Entries and states are compared bit for bit (a NaN with any NaN).
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from test_gpu_compute import _i32

pytestmark = pytest.mark.gpu

INF, NAN = float("inf"), float("nan")


def _same(a: torch.Tensor, b: torch.Tensor) -> bool:
    if a.dtype == torch.uint8:
        return torch.equal(a, b)
    return bool(((a == b) | (a.isnan() & b.isnan())).all())


def _tokens(g, b: int, t: int, ch: int, special: float) -> tuple[torch.Tensor, torch.Tensor]:
    """c, z rows; a share ``special`` of the scores of every other channel is +inf, -inf or NaN."""
    c, z = (torch.randn(b, t, ch, generator=g).to(torch.bfloat16) for _ in range(2))
    kind = torch.randint(0, 8, (b, t, ch), generator=g)
    hit = torch.rand(b, t, ch, generator=g) < special
    hit[:, :, ::2] = False
    for value, kinds in ((INF, (0, 1, 2)), (-INF, (3, 4, 5, 6)), (NAN, (7,))):
        for k in kinds:
            z[hit & (kind == k)] = value
    return c, z


@pytest.mark.parametrize("special", [0.0, 0.3, 0.9])
@pytest.mark.parametrize("fp8", [False, True])
def test_steps_complete_what_a_prompt_left(dev, special, fp8) -> None:
    from saint_kv import ops
    from saint_kv.decode import DecodeCache, LayerSpec

    steps, lens0 = 11, np.array([10, 1, 5, 0, 23])
    b, t, bs = len(lens0), int(lens0.max()) + steps, 16
    cache = DecodeCache([LayerSpec("hca", m=8, fp8=fp8), LayerSpec("csa", m=4, top_k=8, fp8=fp8)], b, 64,
                        block_size=bs, window=8, device=dev)
    g = torch.Generator().manual_seed(int(10 * special) + fp8)
    data = []
    for i, spec in enumerate(cache.layers):
        d = {"kv": torch.randn(b, t, 576, generator=g).to(torch.bfloat16)}
        d["c"], d["z"] = _tokens(g, b, t, 576, special)
        cache.bias[i].copy_(torch.randn(spec.m, 576, generator=g))
        if spec.kind == "csa":
            d["ci"], d["zi"] = _tokens(g, b, t, 128, special)
            cache.idx_bias[i].copy_(torch.randn(spec.m, 128, generator=g))
        data.append({k: v.to(dev) for k, v in d.items()})
    cache.prefill(lens0, data=data)
    at = torch.arange(b, device=dev)
    for s in range(steps):
        for i, d in enumerate(data):
            for k, v in d.items():
                cache.inputs[i][k].copy_(v[at, torch.as_tensor(lens0 + s, device=dev)])
        cache.step()
    cache.check_status()
    done = _i32(lens0 + steps, dev)
    for i, (spec, d) in enumerate(zip(cache.layers, data)):
        bt = cache.groups[cache.group_of_rate[spec.m]].block_table
        for pool, state, bias, c, z in ((cache.pool[i], cache.state[i], cache.bias[i], "c", "z"),
                                        (cache.idx_pool[i], cache.idx_state[i], cache.idx_bias[i], "ci", "zi")):
            if pool is None:
                continue
            want, want_state = torch.zeros_like(pool), torch.zeros_like(state)
            ops.compress_append(want, bt, want_state, d[c], d[z], bias, done, done)
            for q in range(b):
                n = int(lens0[q] + steps)
                for e in range(n // spec.m):
                    page = int(bt[q, e // bs])
                    assert _same(pool[page, e % bs], want[page, e % bs]), (spec.kind, c, q, e)
                if n % spec.m:
                    assert _same(state[q], want_state[q]), (spec.kind, c, q)
