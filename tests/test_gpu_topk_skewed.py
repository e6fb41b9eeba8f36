"""Top-k rows whose scores heap up in a bucket or two: outliers at several
scales, heavy tails, masks of the type's lowest value, ties, values that are not
finite; against the oracle's total order, in the register form and past it.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import reference_cpu as ref

pytestmark = pytest.mark.gpu

LOWEST = np.finfo(np.float32).min


def _scores(kind: str, rows: int, n: int, rng) -> np.ndarray:
    s = rng.standard_normal((rows, n)).astype(np.float32)
    if kind == "relu":
        s = np.maximum(s - 1.5, 0)
    elif kind == "relu_signed_zeros":
        s = np.maximum(s - 1.5, 0) * np.sign(rng.standard_normal((rows, n))).astype(np.float32)
    elif kind == "outliers":  # each level's range is a little of the one before
        for p, x in enumerate((1e4, 1e9, 1e14, 1e19, 1e24, 1e29, 1e34, -1e6, -1e30)):
            s[:, p::n // 3 + 1] = x
    elif kind == "low_outlier":  # all others in a few buckets above the last pick's
        s[:, n // 2] = -500.0
    elif kind == "lowest":
        s[:, : n - n // 5] = LOWEST
    elif kind == "highest":
        s[:, : n // 3] = -LOWEST
    elif kind == "cauchy":
        s = rng.standard_cauchy((rows, n)).astype(np.float32)
    elif kind == "wide":  # every exponent
        s = np.ldexp(s, rng.integers(-149, 125, (rows, n))).astype(np.float32)
    elif kind == "two":
        s = np.where(s > 0.3, np.float32(1), np.nextafter(np.float32(1), np.float32(2)))
    elif kind == "nan":
        s[:, ::2] = np.nan
    elif kind == "inf":
        s[:, ::2], s[:, 1::5] = np.inf, -np.inf
    elif kind == "ninf":
        s[:, 3:] = -np.inf
    elif kind == "ties":
        s = np.round(s * 2)
    return s


KINDS = ("relu", "relu_signed_zeros", "outliers", "low_outlier", "lowest", "highest", "cauchy", "wide", "two", "nan", "inf",
         "ninf", "ties")


@pytest.mark.parametrize("rows,n,k", [(3, 700, 600), (515, 4096, 512), (3, 4096, 2048), (3, 16384, 512), (2, 16384, 2048),
                                      (2, 30000, 1024), (1, 300_000, 2048)])
@pytest.mark.parametrize("kind", KINDS)
def test_skewed_rows(dev, rows, n, k, kind) -> None:
    from saint_kv import ops

    rng = np.random.default_rng(n + k)
    few = min(rows, 3)
    s = np.resize(_scores(kind, few, n, rng), (rows, n))  # rows repeat the first few
    n_valid = np.resize(np.array([n, n - 5, n // 2], dtype=np.int32)[:few], rows)
    out = torch.full((rows, k), 9, dtype=torch.int32, device=dev)
    ops.topk_select(torch.as_tensor(s, device=dev), torch.as_tensor(n_valid, device=dev), n, k, out)
    got = out.cpu().numpy()
    assert np.array_equal(got[:few], ref.topk_select(s[:few], n_valid[:few], k, n))
    assert np.array_equal(got, np.resize(got[:few], got.shape))
