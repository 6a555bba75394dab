"""Plans of the block-size-16 decode kernel: short rows in one launch, head sets
and their rest, and work-item sizes, chosen on the device
from the row lengths: rows around multiples of the 128-token step, launches of
one row up to one past the largest that chooses, empty rows, pages whose
slots bound the item, a workspace of the least size (512-token items) beside
the documented one (128-token items) and none at all where none is needed.
Each against the oracle at 1e-5; a garbage-filled workspace must not show.
"""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from gpu_util import DTYPES, buffer_like
from kvflux_amd import capi, device
from oracle import oracle

pytestmark = pytest.mark.gpu
TOL = 1e-5  # the exact paths' bound: FP32 sums, at most 4 more roundings per chunk merged


def least_bytes(rows, kv_len, q_heads, block_size, head_size):
    """Partials of 512-token items (256 on one-token pages), as documented."""
    item = 256 if block_size == 1 else 512
    chunks = -(-kv_len // item)
    if chunks <= 1:
        return 0
    up = lambda n: (n + 255) // 256 * 256  # noqa: E731
    return up(rows * q_heads * chunks * head_size * 4) + up(rows * q_heads * chunks * 8)


def plan(name, H, Hq, D, bs, rows, kv_len, workspace=1 << 40):
    """(heads per item, heads of a second launch, least item tokens, partial slots)."""
    found = [C.c_uint32(0) for _ in range(4)]
    capi.check(capi.lib().kvflux_paged_attention_plan(H, bs, D, DTYPES[name][0], kv_len, rows, Hq, workspace,
                                                      *map(C.byref, found)))
    return tuple(x.value for x in found)


CASES = [
    # dtype, kv heads, q heads, D, block size, lengths
    ("BFloat16", 8, 32, 128, 16, [127, 128, 129, 1500]),
    ("BFloat16", 2, 8, 128, 16, [300]),
    ("Float16", 2, 8, 128, 16, [1, 80, 128, 17, 0]),  # one item a row, no partials
    ("BFloat16", 2, 14, 64, 4, [129, 200, 2]),
    ("Float16", 4, 28, 128, 16, [0, 1, 640, 641, 2047, 2048, 2049, 4000]),
    ("Float32", 2, 8, 128, 8, [1, 255, 257, 900]),
    ("BFloat16", 1, 4, 64, 1, [1, 256, 257, 400]),
    ("Float16", 1, 11, 64, 64, [20000, 3]),  # a second launch for the heads past the sets
    ("BFloat16", 2, 10, 256, 32, [513, 5000]),
    ("BFloat16", 2, 14, 128, 8, [700, 3]),      # small pages: sets of 5 heads and a launch for the other 2
    ("Float16", 1, 7, 256, 16, [129, 2000]),    # head size 256 the same
    ("Float16", 1, 13, 64, 4, [1000, 513]),     # small pages at 64: 8 and 5
    ("Float32", 1, 11, 128, 8, [1000, 16]),
    ("BFloat16", 1, 2, 64, 16, [1 + 7 * i % 1400 for i in range(256)]),
    ("BFloat16", 1, 2, 64, 16, [1 + 7 * i % 1400 for i in range(257)]),
    ("Float32", 1, 1, 96, 16, [40000, 511, 512, 513]),  # the split kernel's partials, more than 64 of them
    # More than 2048 (row, head) pairs to combine, most of them without partials.
    ("BFloat16", 1, 16, 64, 16, [1 + 13 * i % 300 for i in range(200)] + [5000, 513, 0]),
    ("Float16", 1, 12, 128, 16, [1 + 13 * i % 300 for i in range(300)] + [9000, 0]),  # a fixed item size
    ("BFloat16", 1, 24, 80, 16, [1 + 13 * i % 300 for i in range(100)] + [40000, 512, 513]),
    ("Float16", 2, 20, 256, 32, [1 + 13 * i % 300 for i in range(110)] + [36000]),
]


@pytest.mark.parametrize("case", range(len(CASES)))
def test_item_sizes(gpu, case):
    name, H, Hq, D, bs, lens = CASES[case]
    lib = capi.lib()
    code, host = DTYPES[name]
    lens = np.array(lens, np.uint64)
    rows, max_len = len(lens), int(lens.max())
    width = -(-max_len // bs)
    P = width + 5
    rng = np.random.default_rng(900 + case)
    table = np.stack([rng.permutation(P)[:width] for _ in range(rows)]).astype(np.uint64)
    for r in range(rows):
        table[r, -(-int(lens[r]) // bs):] = 2**64 - 1
    page = H * bs * D
    kc = device.DeviceBuffer(P * page * np.dtype(host).itemsize)
    vc = device.DeviceBuffer(P * page * np.dtype(host).itemsize)
    device.fill_random(kc.ptr, P * page, code, 1, 40 + case)
    device.fill_random(vc.ptr, P * page, code, 1, 80 + case)
    q = oracle.random_elements(0, rows * Hq * D, oracle.F32, 1, 120 + case)
    td, ld, qd = buffer_like(table.reshape(-1)), buffer_like(lens), buffer_like(q)
    live = np.flatnonzero(lens)  # the oracle takes no empty rows
    exp = oracle.paged_attention_rows(kc.download(host), vc.download(host), H, bs, D, code, table[live].reshape(-1),
                                      width, lens[live], q.reshape(rows, -1)[live].reshape(-1), Hq, threads=8)
    full = C.c_size_t(0)
    capi.check(lib.kvflux_paged_attention_workspace_size(rows, max_len, H, Hq, bs, D, C.byref(full)))
    least = least_bytes(rows, max_len, Hq, bs, D)
    assert full.value >= least
    for size in sorted({full.value, least}):
        print(f"items case {case}: workspace {size}", flush=True)
        ws = buffer_like(np.full(size // 4 + 64, -1.0, np.float32))  # -1: the mark that ends a row's partials
        od = buffer_like(np.full(q.size + 8, 7.0, np.float32))
        capi.check(lib.kvflux_paged_attention(kc.ptr, vc.ptr, P, H, bs, D, code, td.ptr, width, ld.ptr, max_len,
                                              rows, Hq, qd.ptr, od.ptr, ws.ptr if size else None, size, None))
        device.synchronize()
        out = od.download(np.float32)
        assert np.all(out[q.size:] == 7.0)
        out = out[:q.size].reshape(rows, -1)
        assert np.all(out[lens == 0] == 0.0)
        assert np.abs(out[live].reshape(-1) - exp).max() < TOL
        assert np.all(ws.download(np.float32)[size // 4:] == -1.0)
    if least > 0:
        status = lib.kvflux_paged_attention(kc.ptr, vc.ptr, P, H, bs, D, code, td.ptr, width, ld.ptr, max_len, rows,
                                            Hq, qd.ptr, qd.ptr, td.ptr, least - 1, None)
        assert status == 1  # KVFLUX_ERR_INVALID_ARGUMENT, before any launch


@pytest.mark.parametrize("name,H,Hq,D,bs", [("BFloat16", 8, 32, 128, 16), ("Float16", 2, 16, 128, 16),
                                             ("BFloat16", 8, 64, 64, 8), ("Float32", 8, 32, 128, 16),
                                             ("BFloat16", 4, 28, 256, 16)])
def test_short_rows_in_one_launch(gpu, name, H, Hq, D, bs):
    """Rows that one 512-token item covers: one launch without partials where
    the combine would cost more than it saves (16-bit caches up to head size
    128: everywhere), the workspace left as it is."""
    lib, code, host = capi.lib(), *DTYPES[name]
    for rows, kv_len in ((1, 130), (1, 256), (8, 400), (32, 512), (100, 300)):
        _, _, item, slots = plan(name, H, Hq, D, bs, rows, kv_len)
        may_split = name == "Float32" or D == 256
        if not may_split or kv_len <= 256 or rows >= 32:
            assert (item, slots) == (-(-kv_len // 128) * 128, 0), (rows, kv_len)
        assert plan(name, H, Hq, D, bs, rows, kv_len, 0)[3] == 0  # nothing without a workspace
        P = rows * -(-kv_len // bs)
        kc = device.DeviceBuffer(P * H * bs * D * np.dtype(host).itemsize)
        vc = device.DeviceBuffer(P * H * bs * D * np.dtype(host).itemsize)
        device.fill_random(kc.ptr, P * H * bs * D, code, 1, 7)
        device.fill_random(vc.ptr, P * H * bs * D, code, 1, 8)
        lens = np.array([1 + (kv_len - 1) * (r + 1) // rows for r in range(rows)], np.uint64)
        table = np.arange(P, dtype=np.uint64).reshape(rows, -1)
        q = oracle.random_elements(0, rows * Hq * D, oracle.F32, 1, 9)
        td, ld, qd = buffer_like(table.reshape(-1)), buffer_like(lens), buffer_like(q)
        full = C.c_size_t(0)
        capi.check(lib.kvflux_paged_attention_workspace_size(rows, kv_len, H, Hq, bs, D, C.byref(full)))
        outs = []
        for size in (full.value, 0):
            ws, od = buffer_like(np.full(size // 4 + 64, 5.0, np.float32)), buffer_like(np.zeros(q.size, np.float32))
            capi.check(lib.kvflux_paged_attention(kc.ptr, vc.ptr, P, H, bs, D, code, td.ptr, table.shape[1], ld.ptr,
                                                  kv_len, rows, Hq, qd.ptr, od.ptr, ws.ptr if size else None, size,
                                                  None))
            device.synchronize()
            outs.append(od.download(np.float32))
            if slots == 0:
                assert np.all(ws.download(np.float32) == 5.0)
        exp = oracle.paged_attention_rows(kc.download(host), vc.download(host), H, bs, D, code, table.reshape(-1),
                                          table.shape[1], lens, q, Hq, threads=8)
        assert max(np.abs(out - exp).max() for out in outs) < TOL
        if slots == 0:
            assert np.array_equal(outs[0], outs[1])


@pytest.mark.parametrize("name,bs,D,cap", [("BFloat16", 16, 256, 5), ("Float16", 8, 128, 5), ("BFloat16", 4, 64, 8),
                                           ("Float32", 8, 128, 8)])
def test_second_launch_only_where_it_saves_head_sets(gpu, name, bs, D, cap):
    """Heads past the last set of `cap` take a launch of their own where that
    saves two sets and the grid is filled; else the sets of the largest divisor
    run in one launch (they share the pages in L2)."""
    for group in range(1, 40):
        sub = next(d for d in range(min(group, cap), 0, -1) if group % d == 0)
        few = plan(name, 1, group, D, bs, 2, 300)
        many = plan(name, 4, 4 * group, D, bs, 64, 16000)
        assert few[:2] == (sub, 0)
        saves = group > cap and sub < 4 and group // sub >= group // cap + 3
        assert many[:2] == ((cap, group % cap) if saves else (sub, 0)), group
