"""The live-page gather around the page sizes where its parts change from
wavefronts of one vector a lane to two and to workgroups: whole outputs of
ragged batches against a numpy restatement of the layout, byte for byte, with a guard past the end.
"""
from __future__ import annotations

import numpy as np
import pytest

from gpu_util import DTYPES, buffer_like
from kvflux_amd import capi, device

pytestmark = pytest.mark.gpu

# kv heads, head size, block size (BF16: head size / 8 vectors a row)
SHAPES = [(1, 8, 1), (1, 56, 9), (1, 64, 8), (5, 104, 1), (1, 64, 16), (3, 344, 1), (2, 64, 32), (7, 584, 1),
          (1, 64, 65), (8, 128, 4), (3, 80, 7), (4, 128, 16)]


@pytest.mark.parametrize("heads,D,bs", SHAPES)
def test_live_gather_page_sizes(gpu, heads, D, bs):
    code, host = DTYPES["BFloat16"]
    lens = np.array([1, 0, bs, bs + 1, 3 * bs - 1 if bs > 1 else 5, 40 * bs, 0, 7], np.uint64)
    pages = -(-lens.astype(np.int64) // bs)
    width, P = int(pages.max()) + 1, int(pages.sum()) + 3
    order = np.random.default_rng(D * bs).permutation(P).astype(np.uint64)
    table = np.full((len(lens), width), 2**64 - 1, np.uint64)
    starts = np.cumsum(pages) - pages
    for r, n in enumerate(pages):
        table[r, :n] = order[starts[r]:starts[r] + n]
    size = P * heads * bs * D
    kc, vc = device.DeviceBuffer(size * 2), device.DeviceBuffer(size * 2)
    device.fill_random(kc.ptr, size, code, 1, 21)
    device.fill_random(vc.ptr, size, code, 1, 22)
    off = (np.cumsum(lens) - lens).astype(np.uint64)
    total = int(lens.sum()) * heads * D
    outs = [buffer_like(np.full(total + 64, 0x7777, np.uint16)) for _ in range(2)]
    td, ld, od, sd = (buffer_like(x) for x in (table.reshape(-1), lens, off, starts.astype(np.uint64)))
    capi.call("kvflux_gather_paged_kv_live", kc.ptr, vc.ptr, P, heads, bs, D, code, td.ptr, width, ld.ptr, od.ptr,
              sd.ptr, len(lens), int(pages.sum()), outs[0].ptr, outs[1].ptr, None)
    device.synchronize()
    for cache, out in zip((kc, vc), outs):
        got, rows = out.download(np.uint16), cache.download(host).reshape(P, heads, bs, D)
        exp = np.concatenate([rows[int(table[r, t // bs]), :, t % bs] for r, n in enumerate(lens) for t in range(int(n))])
        assert np.array_equal(got[:total], exp.reshape(-1).view(np.uint16))
        assert np.all(got[total:] == 0x7777)
