"""Which attention calls take a workgroup per query row, and their results there: a
decode batch with a row per sequence, the drop-in layers' [K | V] rows, more than
two head groups, and both sides of the lines that the route depends on.  A call by
rows leaves the workspace as it is; the split writes it.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import reference_cpu as ref
from test_gpu_attn_rows import ATT_TOL, _want

pytestmark = pytest.mark.gpu


def _cus() -> int:
    return torch.cuda.get_device_properties(0).multi_processor_count


def _check(got: torch.Tensor, want: torch.Tensor) -> None:
    assert bool(torch.isfinite(got).all())
    scale = want.abs().amax(dim=-1, keepdim=True)
    err = (got - want).abs()
    assert bool((err <= ATT_TOL * scale + 1e-4).all()), float((err / (scale + 1e-2)).max())
    assert float(err.mean()) <= 0.1 * ATT_TOL * float(scale.mean()) + 1e-5


def _batch_call(dev, kind, batch, heads, dim, fp8, window=128, top_k=40, m=4, bs=16):
    """(run(workspace) -> output, wanted output) of one query per sequence, lengths 0 and 1 among them."""
    from saint_kv import _lib, ops
    from saint_kv.attention import decode_attention

    g = torch.Generator(device=dev).manual_seed(batch + heads + dim)
    rnd = lambda *s: torch.randn(*s, generator=g, device=dev).to(torch.bfloat16)  # noqa: E731
    lens = np.random.default_rng(batch).integers(2, 260, batch).astype(np.int32)
    lens[:4] = (0, 1, m, 260)
    lens_t = torch.as_tensor(lens, device=dev)
    q, wk, wv = rnd(batch, heads, dim), rnd(batch, window, dim), rnd(batch, window, dim)
    kw = {"sink": torch.randn(heads, generator=g, device=dev)}
    if kind != "swa":
        n_ent = lens // m
        n_max = int(n_ent.max())
        pages = -(-n_max // bs)
        bt = torch.randperm(batch * pages, generator=g, device=dev).view(batch, pages).to(torch.int32)
        cnt = torch.as_tensor(n_ent, device=dev)
        ent = rnd(batch, n_max, dim)
        if fp8:
            pool = torch.zeros(batch * pages, bs, _lib.fp8_entry_bytes(dim), dtype=torch.uint8, device=dev)
            ops.fp8_quant_append(pool, bt, cnt, ent, cnt)
            ent = ref.fp8_unpack_entries(ref.fp8_pack_entries(ent.cpu().view(-1, dim))).view(batch, n_max, dim).to(dev)
        else:
            pool = torch.zeros(batch * pages, bs, dim, dtype=torch.bfloat16, device=dev)
            ops.paged_append(pool, bt, cnt, ent, cnt)
        kw.update(pool=pool, fp8=fp8, block_table=bt, n_entries=cnt, m=m,
                  knorm_w=torch.rand(dim, generator=g, device=dev) + 0.5)
        if kind == "csa":
            kw["picks"] = torch.randint(-1, n_max, (batch, top_k), generator=g, dtype=torch.int32, device=dev)
    want = torch.zeros(batch, heads, dim, dtype=torch.float64, device=dev)
    for b in range(batch):
        n = int(lens[b]) // m
        if lens[b]:
            want[b] = _want(kind, q[b:b + 1], int(lens[b]), wk[b], wv[b], window, kw["sink"], None,
                            ent[b, :n] if kind != "swa" else None, torch.ones(max(n, 1), dtype=torch.bool, device=dev), m,
                            kw["picks"][b:b + 1] if kind == "csa" else None, kw.get("knorm_w"))[0]
    return lambda ws: decode_attention(q, kind, lens_t, wk, wv, workspace=ws, **kw), want


def _run(dev, run, want, by_rows: bool) -> None:
    ws = torch.full((1 << 25,), 12345.0, device=dev)
    got = run(ws)
    assert bool((ws == 12345.0).all()) == by_rows
    _check(got, want)
    assert torch.equal(got, run(ws))  # the same bits again


# items in CUs: heads x dim, whether by rows
@pytest.mark.parametrize("kind,per_cu,more,heads,dim,fp8,by_rows", [
    ("csa", 0.5, -1, 64, 576, False, False), ("csa", 0.5, 0, 64, 576, False, True), ("csa", 0.5, 0, 64, 576, True, False),
    ("hca", 0.5, 0, 16, 576, False, False), ("hca", 0.5, 1, 16, 576, True, True), ("swa", 0.5, 4, 16, 544, False, True),
    ("swa", 1, 1, 16, 576, False, False), ("swa", 1, 1, 64, 384, False, True), ("swa", 0.5, 4, 16, 256, False, False),
    ("swa", 0.5, 4, 40, 160, False, True), ("hca", 1, 1, 8, 128, False, True), ("csa", 1, 1, 8, 512, False, False),
    ("csa", 1.5, 0, 16, 576, False, True), ("csa", 1.5, 0, 16, 576, True, False), ("hca", 1.75, 0, 24, 576, True, True),
    ("hca", 1.5, 0, 16, 160, False, False), ("csa", 0.75, 0, 8, 512, False, True), ("hca", 0.75, 0, 33, 544, False, True),
    ("csa", 0.75, 0, 16, 576, True, True),
])
def test_decode_batches_on_both_sides_of_the_line(dev, kind, per_cu, more, heads, dim, fp8, by_rows) -> None:
    batch = int(per_cu * _cus()) + more
    _run(dev, *_batch_call(dev, kind, batch, heads, dim, fp8), by_rows)


@pytest.mark.parametrize("kind,heads,dim", [("csa", 256, 576), ("hca", 200, 64), ("swa", 192, 512)])
def test_more_than_two_head_groups(dev, kind, heads, dim) -> None:
    groups = -(-heads // 64)
    _run(dev, *_batch_call(dev, kind, _cus() // groups - 3, heads, dim, False), True)


@pytest.mark.parametrize("kind,heads,t_new", [("csa", 64, 150), ("hca", 33, 140), ("swa", 64, 131)])
def test_drop_in_layers_by_rows(dev, kind, heads, t_new) -> None:
    """cached_attention over [K | V] rows of the sequence's whole capacity."""
    from saint_kv import kv_cache as kvc
    from saint_kv.attention import cached_attention

    g = torch.Generator(device=dev).manual_seed(t_new)
    dim, m, window, L, cap = 576, 4, 100, 420, 512
    bf = dict(device=dev, dtype=torch.bfloat16)
    rnd = lambda *s: torch.randn(*s, generator=g, device=dev).to(torch.bfloat16)  # noqa: E731
    mean = lambda x: x.view(1, -1, m, x.shape[-1]).float().mean(2).to(x.dtype)  # noqa: E731
    k, v = rnd(1, L, dim), rnd(1, L, dim)
    top_idx = knorm_w = ent = None
    if kind == "swa":
        layer = kvc.SWAKVCacheLayer(cap, dim, batch_size=1, **bf)
    else:
        h = rnd(1, L, dim)
        ent = mean(h[:, : L // m * m])[0]
        knorm_w = torch.rand(dim, generator=g, device=dev) + 0.5
        if kind == "hca":
            layer = kvc.HCAKVCacheLayer(cap, dim, dim, m, batch_size=1, **bf)
        else:
            layer = kvc.CSAKVCacheLayer(cap, dim, dim, 32, m, batch_size=1, **bf)
            top_idx = torch.randint(-1, L // m, (1, t_new, 48), generator=g, device=dev)
    for at in (slice(0, L - t_new), slice(L - t_new, L)):
        if kind == "swa":
            layer.append(k[:, at], v[:, at])
        elif kind == "hca":
            layer.append(h[:, at], k[:, at], v[:, at], compressor=mean)
        else:
            layer.append(h[:, at], k[:, at], v[:, at], compressor=mean, indexer_compressor=lambda x: mean(x)[..., :32])
    sink = torch.randn(heads, generator=g, device=dev)
    q = rnd(1, heads, t_new, dim)
    assert _cus() / 2 < t_new <= _cus()
    want = _want(kind, q[0].transpose(0, 1), L, k[0], v[0], window, sink, None, ent,
                 torch.ones(L // m, dtype=torch.bool, device=dev), m, None if top_idx is None else top_idx[0], knorm_w)
    _run(dev, lambda ws: cached_attention(layer, q, window=window, top_idx=top_idx, knorm_w=knorm_w, sink=sink,
                                          workspace=ws)[0].transpose(0, 1), want, True)
