"""skv_compress_append_streams: streams of one batch in one launch give the bits
that a call per stream gives, whatever their block lengths, channel counts,
formats and row types, past the streams that one launch takes, and with a
stream that has no rows.
"""

from __future__ import annotations

import pytest
import torch

from test_gpu_compute import _i32

pytestmark = pytest.mark.gpu


def _stream(g, dev, b, t, m, ch, entry, rows):
    from saint_kv._lib import fp8_entry_bytes

    dtype = {"bf16": torch.bfloat16, "f32": torch.float32, "fp8": torch.uint8}[entry]
    n_pages = -(-(t // m + 1) // 16)
    pool = torch.zeros(b * n_pages, 16, fp8_entry_bytes(ch) if entry == "fp8" else ch, dtype=dtype, device=dev)
    c, z = (torch.randn(b, t, ch, generator=g).to(dev, rows) for _ in range(2))
    bt = _i32([[s * n_pages + i for i in range(n_pages)] for s in range(b)], dev)
    return [pool, bt, torch.zeros(b, 3, ch, device=dev), c, z, torch.randn(m, ch, generator=g).to(dev)]


@pytest.mark.parametrize("n_streams", [1, 5, 16, 17, 35])
def test_streams_equal_single_calls(dev, n_streams) -> None:
    from saint_kv import ops

    bf, f32 = torch.bfloat16, torch.float32
    kinds = [(4, 576, "fp8", bf), (4, 128, "bf16", bf), (128, 576, "bf16", bf), (33, 264, "bf16", f32),
             (8, 64, "f32", f32), (1, 8, "bf16", bf), (5, 136, "bf16", bf)]
    g = torch.Generator().manual_seed(n_streams)
    b, lens = 3, [290, 1, 131]
    streams = [_stream(g, dev, b, 290, *kinds[i % len(kinds)]) for i in range(n_streams)]
    if n_streams > 4:  # no rows: nothing changes
        streams[3][3] = streams[3][3][:, :0]
        streams[3][4] = streams[3][4][:, :0]
    single = [[s[0].clone(), s[1], s[2].clone(), *s[3:]] for s in streams]
    # the first call leaves blocks behind, the second completes and leaves others
    for new in (lens, [17, 3, 0]):
        done = lens if new is lens else [x + y for x, y in zip(lens, new)]
        fmts = ops.compress_append_streams([tuple(s) for s in streams], _i32(done, dev), _i32(new, dev))
        assert fmts == [ops.compress_append(*s, _i32(done, dev), _i32(new, dev)) for s in single]
        for i, (s, w) in enumerate(zip(streams, single)):
            assert torch.equal(s[0].view(torch.uint8), w[0].view(torch.uint8)), i
            assert torch.equal(s[2], w[2]), i
            assert (n_streams > 4 and i == 3) or bool(s[0].view(torch.uint8).any()), i


def test_streams_refuse_before_any_launch(dev) -> None:
    from saint_kv import ops

    g = torch.Generator().manual_seed(0)
    good = _stream(g, dev, 2, 8, 4, 64, "bf16", torch.bfloat16)
    bad = _stream(g, dev, 2, 8, 4, 64, "bf16", torch.bfloat16)
    bad[5] = bad[5][:, :32]
    with pytest.raises(ValueError, match="bias"):
        ops.compress_append_streams([tuple(good), tuple(bad)], _i32([8, 8], dev), 8)
    assert not good[0].any()
    assert ops.compress_append_streams([], _i32([8, 8], dev), 8) == []
