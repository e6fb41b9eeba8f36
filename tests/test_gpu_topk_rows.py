"""One workgroup per row: the value-bucket selection of skv_topk_select at the
edges of its sizes (16 scores per thread, 256 and 1024 threads) and on scores
whose buckets it cannot use, against the oracle's total order (score
descending, index ascending, -1 for picks that are not finite).
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import reference_cpu as ref

pytestmark = pytest.mark.gpu


def _scores(kind: str, rows: int, n: int, rng) -> np.ndarray:
    s = rng.standard_normal((rows, n)).astype(np.float32)
    if kind == "equal":  # one bucket
        s[:] = 0.25
    elif kind == "outlier":  # every other score in one bucket
        s[:, n // 2] = 1.0e30
    elif kind == "wide":  # the range overflows fp32
        s[:, 0], s[:, -1] = 3.0e38, -3.0e38
    elif kind == "tiny":  # denormals
        s = (rng.integers(-50, 50, (rows, n)) * 1.0e-44).astype(np.float32)
    elif kind == "ties":
        s = rng.integers(-3, 4, (rows, n)).astype(np.float32)
        s[:, ::7] = -0.0
    elif kind == "nonfinite":
        s[:, 3::11], s[:, 5::13], s[:, 1::17] = np.inf, -np.inf, np.nan
    return s


@pytest.mark.parametrize("rows,n,k", [(3, 1, 1), (3, 5, 2048), (520, 4096, 64), (520, 4097, 64), (2, 4095, 512),
                                      (2, 16384, 1024), (2, 16385, 1024), (1, 40000, 2048)])
@pytest.mark.parametrize("kind", ["normal", "equal", "outlier", "wide", "tiny", "ties", "nonfinite"])
def test_topk_rows(dev, rows, n, k, kind) -> None:
    from saint_kv import ops

    rng = np.random.default_rng(n + k)
    few = min(rows, 3)
    s = np.resize(_scores(kind, few, n, rng), (rows, n))  # rows repeat the first few
    n_valid = np.resize(np.array([n, max(n - 5, 0), n // 3], dtype=np.int32)[:few], rows)
    out = torch.full((rows, k), 9, dtype=torch.int32, device=dev)
    ops.topk_select(torch.as_tensor(s, device=dev), torch.as_tensor(n_valid, device=dev), n, k, out)
    got = out.cpu().numpy()
    want = ref.topk_select(s[:few], n_valid[:few], k, n)
    assert np.array_equal(got[:few, : want.shape[1]], want)
    assert (got[:, want.shape[1]:] == -1).all()
    assert np.array_equal(got, np.resize(got[:few], got.shape))
