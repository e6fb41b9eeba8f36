"""Attention of many query rows: one workgroup per (row, 64 heads) in place of
split units and a merge, taken when the rows fill the device.  Against the
formula in 64 bits at the edges of its tiles, head groups, dims and key runs,
with the tolerance of test_gpu_attention.py (bf16 weights and bf16 partial
outputs).
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import reference_cpu as ref

pytestmark = pytest.mark.gpu

ATT_TOL = 1e-2


def _softmax(s: torch.Tensor, live: torch.Tensor, sink: torch.Tensor | None) -> torch.Tensor:
    """(H, n, k) weights over the live keys (n, k), the sink (H) taking weight; 0 without a live key."""
    s = s.masked_fill(~live[None], -float("inf"))
    if sink is not None:
        s = torch.cat([s, sink[:, None, None].expand(*s.shape[:2], 1)], dim=2)
    mx = s.amax(dim=2, keepdim=True)
    e = torch.exp(s - torch.where(torch.isinf(mx), torch.zeros_like(mx), mx))
    p = (e / e.sum(dim=2, keepdim=True).clamp_min(1e-300))[:, :, : live.shape[1]]
    return torch.where(live.any(1)[None, :, None], p, torch.zeros_like(p))


def _want(kind, q, L, wk, wv, window, sink, softcap, ent, mapped, m, picks, w):
    """One sequence's rows (T, H, D) in 64 bits: its last T of L tokens; mapped: the entries whose page is."""
    t, h, d = q.shape
    dev = q.device
    qq = q.double().transpose(0, 1)
    pos = L - t + torch.arange(t, device=dev)
    at = pos[:, None] - window + 1 + torch.arange(window, device=dev)
    s = torch.einsum("hnd,nkd->hnk", qq, wk.double()[at.clamp_min(0) % wk.shape[0]]) / d ** 0.5
    if softcap:
        s = softcap * torch.tanh(s / softcap)
    sink = sink.double()
    out = torch.einsum("hnk,nkd->hnd", _softmax(s, at >= 0, sink), wv.double()[at.clamp_min(0) % wv.shape[0]])
    if kind != "swa" and len(ent):
        x = ent.double()
        x = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-6) * w.double()
        if kind == "csa":
            live = (picks >= 0) & (picks < len(ent)) & mapped[picks.clamp(0, len(ent) - 1).long()]
            k = x[picks.clamp(0, len(ent) - 1).long()]
            s = torch.einsum("hnd,nkd->hnk", qq, k) / d ** 0.5
            out = out + torch.einsum("hnk,nkd->hnd", _softmax(s, live, None), k)
        else:
            live = (torch.arange(len(ent), device=dev)[None] * m + m - 1 < pos[:, None]) & mapped[None]
            s = torch.einsum("hnd,kd->hnk", qq, x) / d ** 0.5
            out = out + torch.einsum("hnk,kd->hnd", _softmax(s, live, sink), x)
    return out.transpose(0, 1)


@pytest.mark.parametrize("kind,heads,dim,t,window,m,top_k,fp8,softcap", [
    ("csa", 64, 576, 130, 128, 4, 96, False, None), ("csa", 16, 576, 130, 100, 4, 33, True, None),
    ("csa", 80, 64, 129, 31, 4, 600, False, 20.0), ("csa", 8, 512, 140, 1, 4, 1, False, None),
    ("hca", 64, 576, 257, 128, 8, 0, False, None), ("hca", 33, 544, 130, 33, 2, 0, False, 15.0),
    ("hca", 5, 32, 300, 128, 2, 0, False, None), ("hca", 64, 576, 128, 64, 4, 0, True, None),
    ("swa", 64, 576, 300, 128, 1, 0, False, None), ("swa", 70, 96, 140, 97, 1, 0, False, 30.0),
])
def test_attention_by_rows(dev, kind, heads, dim, t, window, m, top_k, fp8, softcap) -> None:
    from saint_kv import _lib, ops
    from saint_kv.attention import decode_attention

    g = torch.Generator(device=dev).manual_seed(heads + dim + t)
    batch, bs, ring = 2, 16, window + t + 3
    lens = np.array([1300 + t, t], dtype=np.int32)  # the second sequence's first queries see little or nothing
    i32 = dict(dtype=torch.int32, device=dev)
    rnd = lambda *s: torch.randn(*s, generator=g, device=dev).to(torch.bfloat16)  # noqa: E731
    # unit variance, as after q_norm: rounding q * w to bf16 moves a score by 2^-9 of its
    # size, and with it its weight, so the tolerance holds for scores of up to about 5
    q, wk, wv = rnd(batch, t, heads, dim), rnd(batch, ring, dim), rnd(batch, ring, dim)
    kw = {"window": window, "sink": torch.randn(heads, generator=g, device=dev), "softcap": softcap}
    lens_t = torch.as_tensor(lens, device=dev)
    if kind != "swa":
        n_ent = lens // m
        n_max = int(n_ent.max())
        pages = -(-n_max // bs) + 1
        table = np.random.default_rng(t).permutation(batch * pages).reshape(batch, pages).astype(np.int32)
        table[0, 1] = -1  # an unmapped page: its entries are not seen
        bt, cnt = torch.as_tensor(table, device=dev), torch.as_tensor(n_ent.astype(np.int32), device=dev)
        ent = rnd(batch, n_max, dim)
        if fp8:
            pool = torch.zeros(batch * pages, bs, _lib.fp8_entry_bytes(dim), dtype=torch.uint8, device=dev)
            ops.fp8_quant_append(pool, bt, cnt, ent, cnt)
            ent = torch.stack([ref.fp8_unpack_entries(ref.fp8_pack_entries(e)) for e in ent.cpu()]).to(dev)
        else:
            pool = torch.zeros(batch * pages, bs, dim, dtype=torch.bfloat16, device=dev)
            ops.paged_append(pool, bt, cnt, ent, cnt)
        kw.update(pool=pool, fp8=fp8, block_table=bt, n_entries=cnt, m=m,
                  knorm_w=torch.rand(dim, generator=g, device=dev) + 0.5)
        if kind == "csa":
            picks = torch.randint(-1, n_max, (batch, t, top_k), generator=g, **i32)
            picks[0, 0] = -1  # a query without picks
            kw["picks"] = picks
    got = decode_attention(q, kind, lens_t, wk, wv, **kw)
    want = torch.empty(batch, t, heads, dim, dtype=torch.float64, device=dev)
    for b in range(batch):
        n = int(lens[b]) // m
        mapped = torch.ones(max(n, 1), dtype=torch.bool, device=dev)
        if b == 0 and kind != "swa":
            mapped[bs: 2 * bs] = False
        want[b] = _want(kind, q[b], int(lens[b]), wk[b], wv[b], window, kw["sink"], softcap,
                        ent[b, :n] if kind != "swa" else None, mapped, m, kw["picks"][b] if kind == "csa" else None,
                        kw.get("knorm_w"))
    assert bool(torch.isfinite(got).all())
    scale = want.abs().amax(dim=-1, keepdim=True)
    err = (got - want).abs()
    assert bool((err <= ATT_TOL * scale + 1e-4).all()), float((err / (scale + 1e-2)).max())
    assert float(err.mean()) <= 0.1 * ATT_TOL * float(scale.mean()) + 1e-5
    assert torch.equal(got, decode_attention(q, kind, lens_t, wk, wv, **kw))  # the same bits again
