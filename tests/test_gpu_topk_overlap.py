"""Score rows that overlap (a stride below the columns, as sliding views have):
the stride does not bound a row's columns."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import reference_cpu as ref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,n,stride", [(1, 20_000, 1), (3, 40_000, 5), (2, 17_000, 16_384), (600, 5_000, 3)])
def test_overlapping_rows(dev, rows, n, stride) -> None:
    from saint_kv import ops

    rng = np.random.default_rng(n)
    base = rng.standard_normal(n + stride * (rows - 1)).astype(np.float32)
    base[-1] = 9.0  # the last row's best is its last column
    scores = torch.as_tensor(base, device=dev).as_strided((rows, n), (stride, 1))
    k = 300
    want = ref.topk_select(np.lib.stride_tricks.sliding_window_view(base, n)[::stride], np.full(rows, n, np.int32), k, n)
    i32 = dict(dtype=torch.int32, device=dev)
    out = torch.full((rows, k), 9, **i32)
    ops.topk_select(scores, torch.full((rows,), n, **i32), torch.full((rows,), n, **i32), k, out)
    assert np.array_equal(out.cpu().numpy(), want)
    ops.topk_select_decode(scores, torch.full((rows,), n + 1, **i32), 1, k, out)  # n visible columns
    assert np.array_equal(out.cpu().numpy(), want)
