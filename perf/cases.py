"""The work that a user of saint-kv has it do, as timed cases.

Seven kinds of call, each through the public Python API:

* ``dropin``  : the reference-shaped cache layers of one request (a prompt
  appended, then tokens one at a time), ``SWAKVCacheLayer`` / ``HCAKVCacheLayer`` /
  ``CSAKVCacheLayer``.
* ``request`` : ``DecodeCache`` takes a batch of finished sequences out, new
  prompts in (``release`` + ``prefill``) and decodes a few steps.
* ``steps``   : a captured run of ``DecodeCache`` steps (``capture`` / ``replay``).
* ``layer``   : one layer of a model's decode step: cache step and attention in
  one call (``step_attend``), with the indexer scores computed in the step.
* ``gather``  : paged append and full gather of raw rows (``ops.decode_append_gather``).
* ``attend``  : attention over the cache, for one query per sequence
  (``decode_attention``) or the tokens of a prompt chunk (``cached_attention``).
* ``topk``    : the indexer's top-k for a chunk of query tokens (``indexer_topk``).

Sizes are those of the repository's benchmark, golden fixtures and tests: rows
of 512 + 64 dims, 64 heads, an indexer of 64 heads x 128, m = 4 and 128,
top-k 512 and 1024, a window of 128, contexts of 1k to 128k tokens, and the
tiny model (head_dim 32, hidden 128).
"""

from __future__ import annotations

import math
import sys
from pathlib import Path

import numpy as np
import torch

_PKG = str(Path(__file__).resolve().parents[1] / "saint-llm_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

BF = torch.bfloat16
F32, F64 = torch.float32, torch.float64
ROPE = 64  # bf16 dims of an fp8 entry


def _dev() -> torch.device:
    return torch.device("cuda", torch.cuda.current_device())


# ---------------------------------------------------------------------------
# The cases
# ---------------------------------------------------------------------------
def listed() -> list[dict]:
    return [
        # the tiny model's three layer kinds on the reference's default dtype:
        # a short prompt and a few greedy tokens (the golden fixtures' shapes)
        {"name": "dropin_tiny", "kind": "dropin", "dtype": "f32", "batch": 2, "dim": 32, "c_idx": 16,
         "hidden": 128, "m_csa": 4, "m_hca": 8, "prompt": 21, "decode": 4},
        # a chat turn: two short prompts replace two finished ones, a few tokens decoded
        {"name": "request_short", "kind": "request", "batch": 2, "lmin": 40, "lmax": 300, "layers": "csa,hca,swa",
         "fp8": False, "m_csa": 4, "m_hca": 128, "top_k": 64, "steps": 3},
        # prompts of a few thousand tokens enter the cache (compression, fp8 quantization, ring)
        {"name": "request_8k", "kind": "request", "batch": 4, "lmin": 6000, "lmax": 8192,
         "layers": "csa,hca,csa8", "fp8": True, "m_csa": 4, "m_hca": 128, "top_k": 512, "steps": 1},
        # the 64k-context decode step of one CSA layer, a captured run of 10 steps
        {"name": "steps_csa_64k", "kind": "steps", "batch": 16, "lmin": 65536, "lmax": 65536, "layers": "csa",
         "m_csa": 4, "m_hca": 128, "top_k": 512, "steps": 10},
        # eight CSA / HCA layers stepped together, ragged 32k - 128k contexts
        {"name": "steps_mixed_8", "kind": "steps", "batch": 32, "lmin": 32768, "lmax": 131072,
         "layers": "csa,hca,csa,hca,csa,hca,csa,hca", "m_csa": 4, "m_hca": 128, "top_k": 512, "steps": 6},
        # one CSA layer of a model's decode step at 64k: scores, step and attention
        {"name": "layer_csa_64k", "kind": "layer", "batch": 16, "lmin": 65536, "lmax": 65536, "heads": 64,
         "idx_heads": 64, "m_csa": 4, "top_k": 512, "fp8": False},
        # raw latent rows: one token per sequence appended, every context gathered
        {"name": "gather_b64", "kind": "gather", "batch": 64, "lmin": 1024, "lmax": 32768, "dim": 576, "block": 64},
        # one decode query per sequence over all compressed entries of an HCA layer
        {"name": "attend_hca_128k", "kind": "attend", "layer": "hca", "batch": 32, "lmin": 32768, "lmax": 131072,
         "t_new": 1, "heads": 64, "dim": 576, "m": 128, "top_k": 0, "fp8": False, "sink": True, "softcap": 0.0},
        # a prompt chunk through a CSA layer: every token over its own picks and its window
        {"name": "prompt_attend_csa", "kind": "attend", "layer": "csa", "batch": 1, "lmin": 16384, "lmax": 16384,
         "t_new": 512, "heads": 64, "dim": 576, "m": 4, "top_k": 512, "fp8": False, "sink": True, "softcap": 0.0},
        # a prompt chunk through an HCA layer: every token over all visible entries and its window
        {"name": "prompt_attend_hca", "kind": "attend", "layer": "hca", "batch": 1, "lmin": 65000, "lmax": 65000,
         "t_new": 1000, "heads": 64, "dim": 576, "m": 128, "top_k": 0, "fp8": False, "sink": True, "softcap": 0.0},
        # the picks of a whole 16k prompt's last chunk
        {"name": "prompt_topk_16k", "kind": "topk", "batch": 1, "offset": 14336, "t_new": 2048, "heads": 64,
         "c": 128, "m": 4, "top_k": 512},
        # two ragged-size chunks at 64k
        {"name": "prompt_topk_64k", "kind": "topk", "batch": 2, "offset": 65000, "t_new": 250, "heads": 64,
         "c": 128, "m": 4, "top_k": 512},
    ]


def _log(rng, lo: float, hi: float) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng) -> dict:
    """One more case of the listed ranges."""
    while True:
        kind = rng.choice(["dropin", "request", "steps", "layer", "gather", "attend", "attend", "topk", "topk"])
        if kind == "dropin":
            c = {"dtype": rng.choice(["f32", "bf16"]), "batch": rng.randint(1, 4),
                 "dim": rng.choice([32, 64, 128, 576]), "c_idx": rng.choice([16, 32, 128]),
                 "hidden": rng.choice([128, 256, 1024]), "m_csa": 4, "m_hca": rng.choice([8, 128]),
                 "prompt": _log(rng, 5, 2000), "decode": rng.randint(1, 6)}
        elif kind == "request":
            top = _log(rng, 30, 8192)
            c = {"batch": _log(rng, 1, 8), "lmin": max(3, int(top * rng.uniform(0.2, 1.0))), "lmax": top,
                 "layers": rng.choice(["csa,hca,swa", "csa", "csa8,hca", "hca", "csa,csa8"]), "fp8": False,
                 "m_csa": 4, "m_hca": rng.choice([32, 128]), "top_k": rng.choice([32, 64, 512]),
                 "steps": rng.randint(0, 4)}
            c["fp8"] = "csa8" in c["layers"]
        elif kind == "steps":
            top = _log(rng, 4096, 131072)
            c = {"batch": _log(rng, 1, 32), "lmin": max(512, int(top * rng.uniform(0.25, 1.0))), "lmax": top,
                 "layers": rng.choice(["csa", "csa,hca", "csa8", "hca,hca", "csa,hca,csa,hca", "csa,swa"]),
                 "m_csa": 4, "m_hca": 128, "top_k": rng.choice([256, 512, 1024]), "steps": rng.choice([3, 6, 10])}
        elif kind == "layer":
            top = _log(rng, 2048, 131072)
            c = {"batch": _log(rng, 1, 32), "lmin": max(512, int(top * rng.uniform(0.25, 1.0))), "lmax": top,
                 "heads": rng.choice([16, 40, 64, 128]), "idx_heads": rng.choice([8, 32, 64]), "m_csa": 4,
                 "top_k": rng.choice([128, 512, 1024]), "fp8": rng.random() < 0.3}
        elif kind == "gather":
            top = _log(rng, 1024, 32768)
            c = {"batch": _log(rng, 4, 64), "lmin": max(256, int(top * rng.uniform(0.05, 1.0))), "lmax": top,
                 "dim": rng.choice([576, 512, 256, 136]), "block": rng.choice([16, 64])}
        elif kind == "attend":
            layer = rng.choice(["csa", "csa", "hca", "hca", "swa"])
            t_new = 1 if rng.random() < 0.4 else _log(rng, 2, 1000)
            top = _log(rng, max(300, t_new), 65536)
            c = {"layer": layer, "batch": _log(rng, 1, 32) if t_new == 1 else rng.randint(1, 2),
                 "lmin": top if t_new > 1 else max(200, int(top * rng.uniform(0.3, 1.0))), "lmax": top,
                 "t_new": t_new, "heads": rng.choice([8, 16, 64, 64, 128]), "dim": rng.choice([64, 128, 512, 576, 576]),
                 "m": 4 if layer == "csa" else rng.choice([32, 128]),
                 "top_k": rng.choice([64, 256, 512]) if layer == "csa" else 0, "fp8": False,
                 "sink": rng.random() < 0.7, "softcap": rng.choice([0.0, 0.0, 30.0])}
            if t_new == 1 and layer != "swa" and c["dim"] == 576:
                c["fp8"] = rng.random() < 0.4
        else:
            t_new = _log(rng, 1, 2048)
            c = {"batch": rng.randint(1, 3), "offset": _log(rng, 16, 65536) - 1, "t_new": t_new,
                 "heads": rng.choice([4, 16, 64, 64]), "c": rng.choice([32, 64, 128, 128]), "m": 4,
                 "top_k": rng.choice([16, 128, 512, 1024])}
        c["kind"] = kind
        if _cost(c) <= 1.0:
            return c


def _cost(c: dict) -> float:
    """A drawn case's work as a share of the largest listed one's (of its kind, or in bytes and flops)."""
    w = work(c)
    if c["kind"] == "topk":
        return w["flops"] / (2.0 * 2048 * 4096 * 64 * 128)
    if c["kind"] == "attend":
        return w["flops"] / (4.0 * 64 * 576 * 1000 * (640 + 2 * 64))
    return max(w["bytes"] / 2.3e9, w["flops"] / 2e11)


# ---------------------------------------------------------------------------
# Shared pieces
# ---------------------------------------------------------------------------
def _lens(case: dict, steps: int = 0) -> np.ndarray:
    """Ragged lengths of the case (fixed by its sizes); after ``steps`` more
    tokens no length is a multiple of 4, so every pooling state is a live one."""
    rng = np.random.default_rng(case["batch"] * 7919 + case["lmax"])
    n = rng.integers(case["lmin"], case["lmax"] + 1, size=case["batch"]).astype(np.int64)
    n[-1] = case["lmax"]
    if steps or case["kind"] == "request":
        n = np.where((n + steps) % 4 == 0, np.maximum(n - 1, 1), n)
        n = np.where((n + steps) % 4 == 0, n + 2, n)
    return n


def _specs(case: dict, idx_heads: int = 0):
    from saint_kv import LayerSpec

    out = []
    for k in case["layers"].split(","):
        if k.startswith("csa"):
            out.append(LayerSpec("csa", m=case["m_csa"], top_k=case["top_k"], fp8=k.endswith("8"), idx_heads=idx_heads))
        else:
            out.append(LayerSpec("hca", m=case["m_hca"]) if k == "hca" else LayerSpec("swa"))
    return out


def _rand(g, *shape, dtype=BF, scale=1.0) -> torch.Tensor:
    t = torch.randn(*shape, generator=g, device=_dev(), dtype=F32)
    return (t if scale == 1.0 else t * scale).to(dtype)


def _entry_bytes(dim: int, fp8: bool) -> int:
    return (dim - ROPE) + (dim - ROPE) // 128 * 4 + 2 * ROPE if fp8 else 2 * dim


class TokenLevelCompressor(torch.nn.Module):
    """A model's compressor as the cache layers are handed it: two projections
    and a positional bias, softmax over every m tokens."""

    def __init__(self, hidden: int, c: int, m: int, g, dtype) -> None:
        super().__init__()
        self.m, self.c = m, c
        self.w_b_kv = torch.nn.Linear(hidden, c, bias=False, device=_dev(), dtype=dtype)
        self.w_b_z = torch.nn.Linear(hidden, c, bias=False, device=_dev(), dtype=dtype)
        self.bias_b = torch.nn.Parameter(_rand(g, m, c, dtype=dtype, scale=0.5))
        with torch.no_grad():
            for w in (self.w_b_kv.weight, self.w_b_z.weight):
                w.copy_(_rand(g, c, hidden, dtype=dtype, scale=hidden ** -0.5))

    def forward(self, h: torch.Tensor) -> torch.Tensor:
        b, t, _ = h.shape
        kv = self.w_b_kv(h).view(b, t // self.m, self.m, self.c)
        z = self.w_b_z(h).view(b, t // self.m, self.m, self.c) + self.bias_b
        return (torch.softmax(z, dim=2) * kv).sum(dim=2)


# ---------------------------------------------------------------------------
# prepare
# ---------------------------------------------------------------------------
def prepare(case: dict, seed: int) -> dict:
    g = torch.Generator(device=_dev()).manual_seed(int(seed))
    with torch.no_grad():
        s = globals()["_prepare_" + case["kind"]](case, g)
    s["case"] = case
    return s


def _dropin_inputs(case: dict, g) -> dict:
    dt = F32 if case["dtype"] == "f32" else BF
    b, n, d, hid = case["batch"], case["prompt"] + case["decode"], case["dim"], case["hidden"]
    s = {"h": _rand(g, b, n, hid, dtype=dt), "k": _rand(g, b, n, d, dtype=dt), "v": _rand(g, b, n, d, dtype=dt)}
    for name, m, c in (("csa", case["m_csa"], d), ("idx", case["m_csa"], case["c_idx"]), ("hca", case["m_hca"], d)):
        s[name] = TokenLevelCompressor(hid, c, m, g, dt)
    return s


def _prepare_dropin(case: dict, g) -> dict:
    from saint_kv import CSAKVCacheLayer, HCAKVCacheLayer, SWAKVCacheLayer

    s = _dropin_inputs(case, g)
    n, dt = case["prompt"] + case["decode"], s["h"].dtype
    kw = dict(batch_size=case["batch"], device=_dev(), dtype=dt)
    s["layers"] = [SWAKVCacheLayer(n, case["dim"], **kw),
                   HCAKVCacheLayer(n, case["hidden"], case["dim"], case["m_hca"], **kw),
                   CSAKVCacheLayer(n, case["hidden"], case["dim"], case["c_idx"], case["m_csa"], **kw)]
    return s


def _request_data(case: dict, g, lens: np.ndarray) -> list[dict]:
    b, t = case["batch"], int(lens.max())
    out = []
    for k in case["layers"].split(","):
        d = {"kv": _rand(g, b, t, 576)}
        if k != "swa":
            d["c"], d["z"] = _rand(g, b, t, 576), _rand(g, b, t, 576)
        if k.startswith("csa"):
            d["ci"], d["zi"] = _rand(g, b, t, 128), _rand(g, b, t, 128)
        out.append(d)
    return out


def _step_inputs(cache, g) -> None:
    """Biases and every input set's new-token rows and scores."""
    for i in range(len(cache.layers)):
        for t in (cache.bias[i], cache.idx_bias[i]):
            if t is not None:
                t.normal_(generator=g)
        for k in range(cache.n_input_sets):
            for t in cache.inputs_by_set[k][i].values():
                t.normal_(generator=g)
            if cache.scores_by_set[k][i] is not None:
                cache.scores_by_set[k][i].normal_(generator=g)


def _prepare_request(case: dict, g) -> dict:
    from saint_kv import DecodeCache

    lens = _lens(case, case["steps"])
    data = _request_data(case, g, lens)
    cache = DecodeCache(_specs(case), case["batch"], int(lens.max()) + case["steps"] + 1, device=_dev(),
                        page_order_seed=None, input_sets=max(1, case["steps"]))
    _step_inputs(cache, g)
    return {"cache": cache, "data": data, "lens": lens}


SLACK = 16384  # tokens a sequence can still take before the batch is replaced


def _tails(cache, g, lens: np.ndarray) -> list:
    """The tokens of every sequence's incomplete blocks."""
    out = []
    for spec in cache.layers:
        t = int((lens % spec.m).max()) if spec.kind != "swa" else 0
        if t == 0:
            out.append(None)
            continue
        d = {n: _rand(g, cache.batch, t, cache.latent) for n in ("c", "z")}
        if spec.kind == "csa":
            d.update({n: _rand(g, cache.batch, t, cache.c_indexer) for n in ("ci", "zi")})
        out.append(d)
    return out


def _prepare_steps(case: dict, g) -> dict:
    from saint_kv import DecodeCache

    n = case["steps"]
    lens = _lens(case, n)
    cache = DecodeCache(_specs(case), case["batch"], int(lens.max()) + SLACK, device=_dev(), input_sets=n)
    _step_inputs(cache, g)
    tails = _tails(cache, g, lens)
    cache.prefill(lens, generator=g, tails=tails)
    torch.cuda.synchronize()
    graph = cache.capture(n)
    return {"cache": cache, "graph": graph, "lens": lens, "tails": tails, "g": g}


def _prepare_layer(case: dict, g) -> dict:
    from saint_kv import DecodeCache, LayerSpec

    lens = _lens(case, 1)
    spec = LayerSpec("csa", m=case["m_csa"], top_k=case["top_k"], fp8=case["fp8"], idx_heads=case["idx_heads"])
    cache = DecodeCache([spec], case["batch"], int(lens.max()) + SLACK, device=_dev(), materialize=False)
    _step_inputs(cache, g)
    cache.inputs[0]["iq"].mul_(0.3)
    cache.inputs[0]["iw"].mul_(case["idx_heads"] ** -0.5)
    tails = _tails(cache, g, lens)
    cache.prefill(lens, generator=g, tails=tails)
    b, h = case["batch"], case["heads"]
    return {"cache": cache, "lens": lens, "tails": tails, "g": g, "q": _rand(g, b, h, 576),
            "knorm_w": torch.rand(576, generator=g, device=_dev()) + 0.5, "sink": _rand(g, h, dtype=F32),
            "v_ring": _rand(g, b, cache.window, 576), "out": torch.zeros(b, h, 576, device=_dev())}


GATHER_STEPS = 512  # tokens per sequence before the batch is replaced


def _prepare_gather(case: dict, g) -> dict:
    from saint_kv import ops

    b, bs, dev = case["batch"], case["block"], _dev()
    lens0 = _lens(case)
    max_pages = int(-(-(int(lens0.max()) + GATHER_STEPS) // bs))
    n_pages = int((-(-(lens0 + GATHER_STEPS) // bs)).sum()) + 7
    i32 = dict(dtype=torch.int32, device=dev)
    s = {"stack": torch.empty(n_pages, **i32), "top": torch.empty(1, **i32),
         "bt": torch.full((b, max_pages), -1, **i32), "lens": torch.zeros(b, **i32),
         "status": torch.zeros(1, **i32), "ones": torch.ones(b, dtype=torch.uint8, device=dev),
         "pool": torch.empty(n_pages, bs, case["dim"], dtype=BF, device=dev).normal_(generator=g),
         "tokens": _rand(g, b, 1, case["dim"]), "units": ops.unit_table(b * max_pages, dev),
         "max_units": b * max_pages, "lens0": torch.as_tensor(lens0.astype(np.int32), device=dev), "done": 0}
    cap = lens0 + GATHER_STEPS
    s["offsets"] = torch.as_tensor(np.concatenate([[0], np.cumsum(cap)[:-1]]), device=dev)
    s["out"] = torch.zeros(int(cap.sum()), case["dim"], dtype=BF, device=dev)
    order = torch.as_tensor(np.random.default_rng(b).permutation(n_pages).astype(np.int32), device=dev)
    ops.free_stack_init(s["stack"], s["top"], order)
    ops.reserve(s["stack"], s["top"], s["bt"], s["lens"], s["lens0"], bs, s["status"])
    return s


def _attend_inputs(case: dict, g) -> dict:
    """Logical contents: entries in order, window rows by position, queries, picks."""
    b, t, h, d = case["batch"], case["t_new"], case["heads"], case["dim"]
    lens = _lens(case)
    n_max = int(lens.max())
    s = {"lens": lens, "q": _rand(g, b, t, h, d), "knorm_w": torch.rand(d, generator=g, device=_dev()) + 0.5,
         "sink": _rand(g, h, dtype=F32) if case["sink"] else None}
    if case["layer"] != "swa":
        s["entries"] = _rand(g, b, max(1, n_max // case["m"]), d)
    if case["layer"] == "csa":  # every query's picks among the entries it sees, best first, -1 where it sees fewer
        q_pos = torch.as_tensor(lens, device=_dev())[:, None] - t + torch.arange(t, device=_dev())
        vis = torch.clamp(q_pos // case["m"], max=s["entries"].shape[1])
        x = torch.rand(b, t, s["entries"].shape[1], generator=g, device=_dev())
        x = x.masked_fill(torch.arange(x.shape[2], device=_dev()) >= vis[:, :, None], -1.0)
        k = min(case["top_k"], x.shape[2])
        v, i = torch.topk(x, k, dim=2)
        s["picks"] = torch.where(v < 0, -1, i)
    rows = n_max if t > 1 else WINDOW
    s["wk"], s["wv"] = _rand(g, b, rows, d), _rand(g, b, rows, d)
    return s


WINDOW = 128


def _prepare_attend(case: dict, g) -> dict:
    from saint_kv import CSAKVCacheLayer, HCAKVCacheLayer, SWAKVCacheLayer, ops

    s = _attend_inputs(case, g)
    b, d, dev, kind = case["batch"], case["dim"], _dev(), case["layer"]
    lens = s["lens"]
    if case["t_new"] > 1:  # the drop-in layer that holds the prompt so far
        n = int(lens[0])
        kw = dict(batch_size=b, device=dev, dtype=BF)
        h = torch.zeros(b, n, 8, dtype=BF, device=dev)
        if kind == "swa":
            s["layer"] = SWAKVCacheLayer(n, d, **kw)
            s["layer"].append(s["wk"], s["wv"])
        elif kind == "hca":
            s["layer"] = HCAKVCacheLayer(n, 8, d, case["m"], **kw)
            s["layer"].append(h, s["wk"], s["wv"], compressor=lambda x: s["entries"])
        else:
            s["layer"] = CSAKVCacheLayer(n, 8, d, 16, case["m"], **kw)
            idx = torch.zeros(b, n // case["m"], 16, dtype=BF, device=dev)
            s["layer"].append(h, s["wk"], s["wv"], compressor=lambda x: s["entries"], indexer_compressor=lambda x: idx)
        s["qt"] = s["q"].transpose(1, 2)
        return s
    s["lens_t"] = torch.as_tensor(lens.astype(np.int32), device=dev)
    s["out"] = torch.zeros(b, case["heads"], d, device=dev)
    if kind != "swa":  # pages of 64 entries
        ent = s["entries"]
        n_ent = (lens // case["m"]).astype(np.int32)
        pages = int(-(-ent.shape[1] // 64))
        n_pages = b * pages
        i32 = dict(dtype=torch.int32, device=dev)
        eb = _entry_bytes(d, case["fp8"])
        pool = torch.zeros(n_pages, 64, eb if case["fp8"] else d, dtype=torch.uint8 if case["fp8"] else BF, device=dev)
        stack, top = torch.empty(n_pages, **i32), torch.empty(1, **i32)
        bt, cnt = torch.full((b, pages), -1, **i32), torch.zeros(b, **i32)
        order = torch.as_tensor(np.random.default_rng(b).permutation(n_pages).astype(np.int32), device=dev)
        ops.free_stack_init(stack, top, order)
        n_t = torch.as_tensor(n_ent, device=dev)
        ops.reserve(stack, top, bt, cnt, n_t, 64)
        (ops.fp8_quant_append if case["fp8"] else ops.paged_append)(pool, bt, cnt, ent, n_t)
        s["kw"] = dict(pool=pool, fp8=case["fp8"], block_table=bt, n_entries=cnt, knorm_w=s["knorm_w"], m=case["m"])
        if kind == "csa":
            s["kw"]["picks"] = s["picks"][:, 0].to(torch.int32).contiguous()
        else:
            s["kw"]["max_entries"] = int(n_ent.max())
    else:
        s["kw"] = {}
    from saint_kv.attention import decode_attention, last_workspace

    _decode_attend(s, case, decode_attention, None)
    s["ws"] = last_workspace()  # kept by the program for its later calls
    return s


def _topk_inputs(case: dict, g) -> dict:
    b, t, h, c = case["batch"], case["t_new"], case["heads"], case["c"]
    n = (case["offset"] + t) // case["m"]
    return {"q": _rand(g, b, t, h, c, scale=0.3), "w": _rand(g, b, t, h, dtype=F32, scale=h ** -0.5),
            "k": _rand(g, b, max(n, 1), c), "n": n}


def _prepare_topk(case: dict, g) -> dict:
    return _topk_inputs(case, g)


# ---------------------------------------------------------------------------
# run
# ---------------------------------------------------------------------------
def run(state: dict):
    return globals()["_run_" + state["case"]["kind"]](state, state["case"])


def _run_dropin(s: dict, case: dict):
    swa, hca, csa = s["layers"]
    p, n = case["prompt"], case["prompt"] + case["decode"]
    out = None
    with torch.no_grad():
        for layer in s["layers"]:
            layer.reset()
        for lo, hi in [(0, p)] + [(i, i + 1) for i in range(p, n)]:
            h, k, v = s["h"][:, lo:hi], s["k"][:, lo:hi], s["v"][:, lo:hi]
            out = [swa.append(k, v), hca.append(h, k, v, compressor=s["hca"]),
                   csa.append(h, k, v, compressor=s["csa"], indexer_compressor=s["idx"])]
    return out


def _run_request(s: dict, case: dict):
    cache = s["cache"]
    live = cache.host_lens > 0
    if live.any():
        cache.release(live)
    cache.prefill(s["lens"], data=s["data"])
    for k in range(case["steps"]):
        cache.step(k)
    return {"pool": cache.pool, "idx_pool": cache.idx_pool, "state": cache.state, "ring": cache.ring,
            "lens": cache.tok_lens, **({"topk": cache.topk_idx, "window": cache.out_window,
                                        "entries": [e for e, sp in zip(cache.out_entries, cache.layers) if sp.kind == "csa"]}
                                       if case["steps"] else {})}


def _replace(s: dict) -> None:
    """The batch has reached the end of its slots: new sequences take its place."""
    cache = s["cache"]
    cache.release(np.ones(cache.batch, dtype=bool))
    cache.prefill(s["lens"], generator=s["g"], tails=s["tails"])


def _run_steps(s: dict, case: dict):
    cache = s["cache"]
    if int(cache.host_lens.max()) + case["steps"] > cache.max_len:
        _replace(s)
    s["graph"].replay()
    return {"topk": cache.topk_idx, "window": cache.out_window, "state": cache.state, "idx_state": cache.idx_state,
            "entries": [e for e, sp in zip(cache.out_entries, cache.layers) if sp.kind == "csa"],
            "lens": cache.tok_lens}


def _run_layer(s: dict, case: dict):
    cache = s["cache"]
    if int(cache.host_lens.max()) + 1 > cache.max_len:
        _replace(s)
    out = cache.step_attend(s["q"], s["knorm_w"], sink=s["sink"], v_ring=s["v_ring"], out=s["out"])
    return {"out": out, "topk": cache.topk_idx[0], "state": cache.state[0], "lens": cache.tok_lens}


def _run_gather(s: dict, case: dict):
    from saint_kv import ops

    if s["done"] == GATHER_STEPS:  # every sequence has filled its slot: the next batch takes the pages
        ops.release(s["stack"], s["top"], s["bt"], s["lens"], s["ones"], case["block"], s["status"])
        ops.reserve(s["stack"], s["top"], s["bt"], s["lens"], s["lens0"], case["block"], s["status"])
        s["done"] = 0
    s["done"] += 1
    return ops.decode_append_gather(s["stack"], s["top"], s["bt"], s["lens"], s["pool"], s["tokens"], 1, s["out"],
                                    s["units"], s["max_units"], s["offsets"], s["status"])


def _decode_attend(s: dict, case: dict, fn, ws):
    return fn(s["q"][:, 0], case["layer"], s["lens_t"], s["wk"], s["wv"], sink=s["sink"],
              softcap=case["softcap"] or None, out=s["out"], workspace=ws, window=WINDOW, **s["kw"])


def _run_attend(s: dict, case: dict):
    from saint_kv.attention import cached_attention, decode_attention

    if case["t_new"] == 1:
        return _decode_attend(s, case, decode_attention, s["ws"])
    kw = {"top_idx": s["picks"]} if case["layer"] == "csa" else {}
    if case["layer"] != "swa":
        kw["knorm_w"] = s["knorm_w"]
    return cached_attention(s["layer"], s["qt"], window=WINDOW, sink=s["sink"], softcap=case["softcap"] or None, **kw)


def _run_topk(s: dict, case: dict):
    from saint_kv.indexer import indexer_topk

    return indexer_topk(s["q"], s["w"], s["k"], cache_offset=case["offset"], total_len=case["offset"] + case["t_new"],
                        n_blocks=s["n"], m=case["m"], top_k=case["top_k"])


# ---------------------------------------------------------------------------
# work
# ---------------------------------------------------------------------------
def _step_bytes(case: dict, lens: np.ndarray, materialize: bool = True) -> float:
    """One step of the case's layers at token counts ``lens``: new rows in and
    ring, state read and written, scores read, picks and dense entries gathered."""
    b, e, total = len(lens), 2 * 576, 0.0
    win = float(np.minimum(lens, WINDOW).sum())
    for k in case["layers"].split(","):
        total += 2 * b * e + (2 * win * e if materialize else 0)
        if k == "swa":
            continue
        m = case["m_csa"] if k.startswith("csa") else case["m_hca"]
        eb = _entry_bytes(576, k.endswith("8"))
        total += b * (2 * e + 6 * 576 * 4 + 576 * 4 + eb / m)
        if k == "hca":
            total += float((lens // m).sum()) * 2 * e if materialize else 0.0
        else:
            total += b * (4 * 128 + 6 * 128 * 4 + 128 * 4 + 256 / m)
            sel = float(np.minimum(lens // m, case["top_k"]).sum())
            total += float((lens // m).sum()) * 4 + b * case["top_k"] * 4 + (sel * (eb + e) if materialize else 0)
    return total


def _attend_flops(case: dict, lens: np.ndarray) -> tuple[float, float]:
    """(multiply-adds x 2 of both products over the visible keys, distinct keys' bytes)."""
    t, h, d = case["t_new"], case["heads"], case["dim"]
    keys = rows = 0.0
    for n in lens:
        q = np.arange(n - t, n)
        win = np.minimum(q + 1, WINDOW)
        keys += float(win.sum())
        rows += min(int(n), WINDOW + t - 1) * 4 * d
        if case["layer"] != "swa":
            vis = q // case["m"]
            if case["layer"] == "csa":
                picked = np.minimum(vis, case["top_k"])
                keys += float(picked.sum())
                rows += min(float(picked.sum()), int(n) // case["m"]) * _entry_bytes(d, case["fp8"]) + 4 * t * case["top_k"]
            else:
                keys += float(vis.sum())
                rows += int(vis.max()) * _entry_bytes(d, case["fp8"])
    return 4.0 * h * d * keys, rows


def work(case: dict) -> dict:
    k = case["kind"]
    if k == "dropin":
        es = 4 if case["dtype"] == "f32" else 2
        b, n, d, hid = case["batch"], case["prompt"] + case["decode"], case["dim"], case["hidden"]
        cols = 2 * (2 * d + case["c_idx"])  # two projections of three streams
        ent = n // case["m_csa"] * (d + case["c_idx"]) + n // case["m_hca"] * d
        return {"bytes": float(es * (b * n * hid + cols * hid + b * (3 * 4 * n * d + 2 * ent))),
                "flops": 2.0 * b * n * hid * cols}
    if k == "request":
        lens = _lens(case, case["steps"])
        total = 0.0
        for lay in case["layers"].split(","):
            total += float(np.minimum(lens, WINDOW).sum()) * 4 * 576
            if lay != "swa":
                m = case["m_csa"] if lay.startswith("csa") else case["m_hca"]
                total += float(lens.sum()) * (4 * 576 + _entry_bytes(576, lay.endswith("8")) / m)
                if lay.startswith("csa"):
                    total += float(lens.sum()) * (4 * 128 + 256 / m)
        total += sum(_step_bytes(case, lens + i + 1) for i in range(case["steps"]))
        return {"bytes": total, "flops": 8.0 * total / 4}
    if k == "steps":
        lens = _lens(case, case["steps"])
        return {"bytes": sum(_step_bytes(case, lens + i + 1) for i in range(case["steps"])), "flops": 0.0}
    if k == "layer":
        lens = _lens(case, 1) + 1
        c = dict(case, layers="csa8" if case["fp8"] else "csa")
        n_ent = float((lens // case["m_csa"]).sum())
        keys = float(np.minimum(lens // case["m_csa"], case["top_k"]).sum())
        win = float(np.minimum(lens, WINDOW).sum())
        return {"bytes": _step_bytes(c, lens, False) + n_ent * 256 + keys * _entry_bytes(576, case["fp8"]) +
                win * 4 * 576 + len(lens) * (case["heads"] * 576 * 6 + case["idx_heads"] * 260),
                "flops": 2.0 * n_ent * case["idx_heads"] * 128 + 4.0 * case["heads"] * 576 * (keys + win)}
    if k == "gather":
        lens, e = _lens(case) + 1, 2 * case["dim"]
        return {"bytes": float(lens.sum()) * 2 * e + len(lens) * 2 * e + float((-(-lens // case["block"])).sum()) * 4,
                "flops": 0.0}
    if k == "attend":
        lens = _lens(case)
        flops, rows = _attend_flops(case, lens)
        return {"bytes": rows + len(lens) * case["t_new"] * case["heads"] * case["dim"] * 6.0, "flops": flops}
    b, t, h, c, m = case["batch"], case["t_new"], case["heads"], case["c"], case["m"]
    n = (case["offset"] + t) // m
    vis = float(np.minimum(np.arange(case["offset"], case["offset"] + t) // m, n).sum())
    return {"bytes": b * (n * c * 2.0 + t * h * (2.0 * c + 4) + t * min(case["top_k"], n) * 8.0),
            "flops": max(1.0, 2.0 * b * vis * h * c)}


# ---------------------------------------------------------------------------
# tolerance
# ---------------------------------------------------------------------------
def tolerance(case: dict):
    k = case["kind"]
    if k == "gather":
        return "exact"
    if k == "dropin":  # fp32: projections and pooling in fp32; bf16: rounded projections
        return {"rel": 1e-5, "max": 1e-4} if case["dtype"] == "f32" else {"rel": 1e-2, "max": 4e-2}
    if k == "request":  # pooled in fp32, one rounding to bf16 (then perhaps to an fp8 code)
        return {"rel": 2e-3, "max": 1e-2, "differ": 2e-3}
    if k == "steps":  # fp32 states; the entries are copies, of rows pooled and rounded to bf16 once
        return {"rel": 1e-4, "max": 1e-2, "differ": 0.0}
    if k == "layer":
        return {"rel": 1e-2, "max": 8e-2, "differ": 1e-2}
    if k == "attend":  # bf16 weights and partial outputs: 2.4e-3 off the 64-bit result
        return {"rel": 1e-2, "max": 8e-2}
    return {"differ": 1e-2}  # picks: neighbours whose fp32 scores are closer than the sums' rounding trade places


# ---------------------------------------------------------------------------
# exact: the same in 64 bits, in plain torch
# ---------------------------------------------------------------------------
def exact(case: dict, seed: int):
    g = torch.Generator(device=_dev()).manual_seed(int(seed))
    f = globals().get("_exact_" + case["kind"])
    with torch.no_grad():
        return None if f is None else f(case, g)


def _pool64(c, z, bias, m):
    """(B, n // m, C) pooled entries of tokens (B, n, C), n a multiple of m."""
    b, n, ch = c.shape
    v = z.reshape(b, n // m, m, ch) + bias
    return (torch.softmax(v, dim=2) * c.reshape(b, n // m, m, ch)).sum(dim=2)


def _state64(c, z, bias):
    """(B, 3, C): max, sum of weights and weighted sum over tokens (B, r, C)."""
    v = z + bias[: z.shape[1]]
    mx = v.amax(dim=1, keepdim=True)
    w = torch.exp(v - mx)
    return torch.stack([mx[:, 0], w.sum(1), (w * c).sum(1)], dim=1)


def _exact_dropin(case: dict, g):
    s = _dropin_inputs(case, g)
    n = case["prompt"] + case["decode"]
    h, k, v = (s[x].double() for x in ("h", "k", "v"))

    def entries(name, m):
        comp = s[name]
        p = n // m * m
        c, z = (h[:, :p] @ w.weight.double().t() for w in (comp.w_b_kv, comp.w_b_z))
        return _pool64(c, z, comp.bias_b.double(), m)

    return [(k, v), (entries("hca", case["m_hca"]), k, v),
            (entries("csa", case["m_csa"]), entries("idx", case["m_csa"]), k, v)]


def _exact_request(case: dict, g):
    """States, rings and bf16 pools after the first pass (pages are handed out in order)."""
    from types import SimpleNamespace

    lens = _lens(case, case["steps"])
    data = _request_data(case, g, lens)
    b, n, steps = case["batch"], int(lens.max()), case["steps"]
    max_len, kinds = int(lens.max()) + steps + 1, case["layers"].split(",")
    # the biases and input sets, drawn as prepare draws them
    zeros = lambda *sh: torch.zeros(*sh, dtype=BF, device=_dev())  # noqa: E731
    cache = SimpleNamespace(layers=kinds, n_input_sets=max(1, steps), bias=[], idx_bias=[], inputs_by_set=[[] for _ in range(max(1, steps))],
                            scores_by_set=[[] for _ in range(max(1, steps))])
    for kd in kinds:
        m = case["m_csa"] if kd.startswith("csa") else case["m_hca"]
        cache.bias.append(None if kd == "swa" else torch.zeros(m, 576, device=_dev()))
        cache.idx_bias.append(torch.zeros(m, 128, device=_dev()) if kd.startswith("csa") else None)
        for k in range(max(1, steps)):
            d = {"kv": zeros(b, 576)}
            if kd != "swa":
                d["c"], d["z"] = zeros(b, 576), zeros(b, 576)
            if kd.startswith("csa"):
                d["ci"], d["zi"] = zeros(b, 128), zeros(b, 128)
            cache.inputs_by_set[k].append(d)
            cols = -(-max(1, max_len // m) // 4) * 4
            cache.scores_by_set[k].append(torch.zeros(b, cols, device=_dev()) if kd.startswith("csa") else None)
    _step_inputs(cache, g)
    out = {"pool": [], "idx_pool": [], "state": [], "ring": [], "lens": None}
    for i, kd in enumerate(kinds):
        ring = torch.zeros(b, WINDOW, 576, dtype=F64, device=_dev())

        def tokens(name, j, i=i):
            """Sequence j's rows of one input stream: its prompt, then the steps' tokens."""
            new = [cache.inputs_by_set[k][i][name][j:j + 1] for k in range(steps)]
            return torch.cat([data[i][name][j, : lens[j]], *new]).double()

        for j in range(b):
            kv = tokens("kv", j)
            pos = torch.arange(max(0, len(kv) - WINDOW), len(kv), device=_dev())
            ring[j, pos % WINDOW] = kv[pos]
        out["ring"].append(ring)
        if kd == "swa":
            for name in ("pool", "idx_pool", "state"):
                out[name].append(None)
            continue
        m = case["m_csa"] if kd.startswith("csa") else case["m_hca"]
        stride = max(1, -(-(max_len // m) // 64))
        table = [list() for _ in range(b)]  # pages pop in ascending order
        nxt = 0
        for j in range(b):
            for _ in range(-(-(int(lens[j]) // m) // 64)):
                table[j].append(nxt)
                nxt += 1
        for st in range(steps):
            for j in range(b):
                if -(-((int(lens[j]) + st + 1) // m) // 64) > len(table[j]):
                    table[j].append(nxt)
                    nxt += 1
        for pool, ck, zk, ch, bias in (("pool", "c", "z", 576, cache.bias[i]), ("idx_pool", "ci", "zi", 128, cache.idx_bias[i])):
            if pool == "idx_pool" and kd == "hca":
                out[pool].append(None)
                continue
            if pool == "pool":
                out["state"].append(torch.zeros(b, 3, 576, dtype=F64, device=_dev()))
            p = torch.zeros(b * stride * 64, ch, dtype=F64, device=_dev())
            for j in range(b):
                c, z = tokens(ck, j), tokens(zk, j)
                e = len(c) // m
                if e:
                    at = torch.as_tensor(table[j], device=_dev())[torch.arange(e, device=_dev()) // 64] * 64 + torch.arange(e, device=_dev()) % 64
                    p[at] = _pool64(c[None, : e * m], z[None, : e * m], bias.double(), m)[0]
                if pool == "pool" and len(c) % m:
                    out["state"][-1][j] = _state64(c[None, e * m:], z[None, e * m:], bias.double())[0]
            out[pool].append(None if kd.endswith("8") and pool == "pool" else p.view(b * stride, 64, ch))
    return out


def _exact_layer(case: dict, g):
    """The first pass: scores, picks and attention of every sequence's new token."""
    if case["fp8"]:
        return None
    dev, lens, m, b, h, ih = _dev(), _lens(case, 1), case["m_csa"], case["batch"], case["heads"], case["idx_heads"]
    f32 = lambda *sh: torch.zeros(*sh, device=dev).normal_(generator=g)  # noqa: E731
    bf = lambda *sh: torch.zeros(*sh, dtype=BF, device=dev).normal_(generator=g)  # noqa: E731
    max_len = int(lens.max()) + SLACK
    n_ent = max_len // m
    stride = max(1, -(-n_ent // 64))
    n_pages = b * stride
    # drawn in the order prepare draws them
    bias, _ = f32(m, 576), f32(m, 128)
    kv, c, z, _, _, iq = bf(b, 576), bf(b, 576), bf(b, 576), bf(b, 128), bf(b, 128), bf(b, ih, 128).mul_(0.3)
    iw = f32(b, ih).mul_(ih ** -0.5)
    f32(b, -(-n_ent // 4) * 4)
    t = int((lens % m).max())
    tails = [_rand(g, b, t, ch) for ch in (576, 576, 128, 128)] if t else None
    ring = bf(b, WINDOW, 576)
    pool, idx = (torch.zeros(n_pages, 64, ch, dtype=BF, device=dev) for ch in (576, 128))
    for p in (pool, idx):
        for chunk in p.split(4096):
            chunk.normal_(generator=g)
    q, knorm_w = _rand(g, b, h, 576).double(), (torch.rand(576, generator=g, device=dev) + 0.5).double()
    sink, v_ring = _rand(g, h, dtype=F32).double()[:, None], _rand(g, b, WINDOW, 576).double()
    order = torch.as_tensor(np.random.default_rng(0).permutation(n_pages), device=dev)
    out = torch.zeros(b, h, 576, dtype=F64, device=dev)
    state, at = torch.zeros(b, 3, 576, dtype=F64, device=dev), 0
    for j in range(b):
        n = int(lens[j])
        pages = order[at: at - (-(n // m) // 64)]
        at += len(pages)
        keys = idx[pages].view(-1, 128)[: n // m].double()
        sc = iw[j].double() @ torch.relu(iq[j].double() @ keys.t())
        top = torch.sort(sc, descending=True, stable=True)[1][: case["top_k"]]
        x = pool[pages].view(-1, 576)[top].double()
        x = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-6) * knorm_w
        wk = ring[j].double()
        wk[n % WINDOW] = kv[j].double()
        out[j] = _softmax64(q[j] @ x.t() / 24.0, None) @ x + _softmax64(q[j] @ wk.t() / 24.0, sink) @ v_ring[j]
        r = n % m  # the incomplete block before the new token
        cz = [torch.cat(([tl[j, :r]] if r else []) + [new[j:j + 1]]).double()[None] for tl, new in
              zip(tails[:2] if tails else (None, None), (c, z))]
        state[j] = _state64(cz[0], cz[1], bias.double())[0]
    return {"out": out, "topk": None, "state": state, "lens": None}


def _softmax64(s, sink):
    """softmax over the last dim with an extra logit per head that takes weight but has no value."""
    if sink is not None:
        s = torch.cat([s, sink.expand(*s.shape[:-1], 1)], dim=-1)
    mx = s.amax(dim=-1, keepdim=True)
    mx = torch.where(torch.isinf(mx), torch.zeros_like(mx), mx)
    e = torch.exp(s - mx)
    p = e / e.sum(dim=-1, keepdim=True).clamp_min(1e-300)
    return p[..., :-1] if sink is not None else p


def _exact_attend(case: dict, g):
    if case["fp8"]:
        return None
    s = _attend_inputs(case, g)
    b, t, h, d = case["batch"], case["t_new"], case["heads"], case["dim"]
    lens, dev = s["lens"], _dev()
    q = s["q"].double()
    sink = s["sink"].double()[:, None, None] if s["sink"] is not None else None  # (H, 1, 1)
    out = torch.zeros(b, t, h, d, dtype=F64, device=dev)
    wk, wv = s["wk"].double(), s["wv"].double()
    kn = None
    if case["layer"] != "swa":
        x = s["entries"].double()
        kn = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-6) * s["knorm_w"].double()
    inf = float("inf")
    for j in range(b):
        for lo in range(0, t, 64):
            hi = min(t, lo + 64)
            pos = int(lens[j]) - t + torch.arange(lo, hi, device=dev)  # the queries' positions
            qq = q[j, lo:hi].transpose(0, 1)  # (H, n, d)
            # window
            at = pos[:, None] - WINDOW + 1 + torch.arange(WINDOW, device=dev)
            row = at.clamp_min(0) % wk.shape[1]
            sc = torch.einsum("hnd,nkd->hnk", qq, wk[j][row]) / math.sqrt(d)
            if case["softcap"]:
                sc = case["softcap"] * torch.tanh(sc / case["softcap"])
            sc = sc.masked_fill((at < 0)[None], -inf)
            o = torch.einsum("hnk,nkd->hnd", _softmax64(sc, sink), wv[j][row])
            if case["layer"] == "csa":
                pk = s["picks"][j, lo:hi]
                kk = kn[j][pk.clamp_min(0)]
                sc = torch.einsum("hnd,nkd->hnk", qq, kk) / math.sqrt(d)
                sc = sc.masked_fill((pk < 0)[None], -inf)
                o = o + torch.einsum("hnk,nkd->hnd", _softmax64(sc, None), kk)
            elif case["layer"] == "hca":
                vis = torch.arange(kn.shape[1], device=dev)[None] * case["m"] + case["m"] - 1 < pos[:, None]
                sc = torch.einsum("hnd,kd->hnk", qq, kn[j]) / math.sqrt(d)
                sc = sc.masked_fill(~vis[None], -inf)
                p = _softmax64(sc, sink)
                o = o + torch.where(vis.any(1)[None, :, None], torch.einsum("hnk,kd->hnd", p, kn[j]), 0.0)
            out[j, lo:hi] = o.transpose(0, 1)
    return out[:, 0] if t == 1 else out.transpose(1, 2)


def _exact_steps(case: dict, g):
    return None  # copies and whole values; the pooling is the request cases' (checked there in 64 bits)


def _exact_topk(case: dict, g):
    return None  # whole values
