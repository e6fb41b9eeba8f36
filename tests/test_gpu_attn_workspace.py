"""The attention's workspace over the number of rows: a call by rows asks for no
more than the split calls of fewer rows, and a workspace of the most rows serves
every smaller call.
"""

from __future__ import annotations

import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["swa", "hca", "csa"])
@pytest.mark.parametrize("heads,dim,fp8", [(64, 576, False), (64, 576, True), (16, 576, False), (16, 576, True), (128, 512, False),
                                           (16, 160, False), (8, 128, False), (80, 544, False)])
def test_workspace_over_rows(dev, kind, heads, dim, fp8) -> None:
    from saint_kv import _lib
    from saint_kv.attention import KIND, AttentionDesc

    if fp8 and kind == "swa":
        pytest.skip("no entries")
    d = AttentionDesc()
    d.kind, d.format = KIND[kind], _lib.SKV_FMT_FP8 if fp8 else _lib.SKV_FMT_BF16
    d.n_heads, d.head_dim, d.window, d.batch = heads, dim, 128, 1
    d.entry_bytes = _lib.fp8_entry_bytes(dim) if fp8 else 2 * dim
    d.block_size, d.n_pages, d.bt_stride, d.m = 64, 4096, 64, 4
    d.top_k = d.pick_stride = 512

    def need(rows: int) -> int:
        d.batch = rows
        n = int(_lib.load().skv_attention_workspace(ctypes.byref(d)))
        assert n >= 0
        return n

    most = 16384
    sizes = [need(r) for r in range(1, 2100)]
    assert all(n <= need(most) for n in sizes)
    unit = 64 * (8 + 2 * dim)
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    units = need(most) // unit
    groups = -(-heads // 64)
    if kind == "swa" and dim > 128 and heads < 48 * groups:
        assert units == most * groups  # split at many rows, a unit each
    elif heads in (64, 128) or dim == 128 or kind == "swa":
        assert units <= 3 * cus // 2
    else:
        assert units <= 13 * cus
