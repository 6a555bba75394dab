"""Prefill launches whose wavefronts split the keys of a workgroup (small
grids): rows whose only keys lie in one half of a tile, last tiles with one or
both halves live, groups at and past the halved row count, every dtype and
head size, key splits beside them, and rows in different sequences of one
batch. FP32 caches and the exact path at 1e-5 against the oracle over whole
outputs, the rounded path at 2e-2.
"""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from gpu_util import DTYPES, buffer_like
from kvflux_amd import capi, device
from oracle import oracle

pytestmark = pytest.mark.gpu


def arena(name, kv_heads, bs, head_size, kv_lens, seed):
    """Random pages for every sequence: (k, v, pages, table, width)."""
    code, host = DTYPES[name]
    width = max(-(-int(n) // bs) for n in kv_lens) + 1
    blocks = len(kv_lens) * width + 2
    page = kv_heads * bs * head_size
    kc = device.DeviceBuffer(blocks * page * np.dtype(host).itemsize)
    vc = device.DeviceBuffer(blocks * page * np.dtype(host).itemsize)
    device.fill_random(kc.ptr, blocks * page, code, 1, seed)
    device.fill_random(vc.ptr, blocks * page, code, 1, seed + 1)
    order = np.random.default_rng(seed).permutation(blocks).astype(np.uint64)
    table = np.full((len(kv_lens), width), 2**64 - 1, np.uint64)
    for i, n in enumerate(kv_lens):
        pages = -(-int(n) // bs)
        table[i, :pages] = order[i * width:i * width + pages]
    return kc, vc, blocks, table, width


BATCH = [  # name, kv heads, q heads, D, block size, (kv, queries) of each sequence
    ("BFloat16", 2, 8, 128, 16, [(1, 1), (31, 31), (33, 33), (64, 64), (65, 65)]),
    ("Float16", 1, 4, 128, 8, [(97, 97), (320, 1), (352, 40), (130, 130)]),  # rows starting in either half
    ("BFloat16", 1, 128, 128, 16, [(70, 70)]),   # a group of exactly half the rows (one token a workgroup)
    ("BFloat16", 1, 129, 128, 16, [(70, 70)]),   # one past it
    ("Float16", 2, 6, 64, 1, [(200, 200), (63, 5)]),
    ("BFloat16", 1, 3, 256, 32, [(129, 129), (512, 33)]),
    ("Float32", 2, 8, 128, 16, [(1, 1), (32, 32), (33, 33), (300, 300), (161, 7)]),
    ("Float32", 1, 64, 64, 16, [(96, 96)]),
    ("Float32", 1, 65, 64, 4, [(96, 96)]),
]


@pytest.mark.parametrize("case", range(len(BATCH)))
def test_batch_key_parts(gpu, case):
    name, kv_heads, q_heads, D, bs, seqs = BATCH[case]
    code, host = DTYPES[name]
    kv = np.array([a for a, _ in seqs], np.uint64)
    ql = np.array([b for _, b in seqs], np.uint64)
    off = np.concatenate([[0], np.cumsum(ql)[:-1]]).astype(np.uint64)
    kc, vc, blocks, table, width = arena(name, kv_heads, bs, D, kv, 700 + 2 * case)
    total, row = int(ql.sum()), q_heads * D
    q = oracle.random_elements(0, total * row, oracle.F32, 1, 750 + case)
    td, qd, kd, ld, sd = (buffer_like(x) for x in (table.reshape(-1), q, kv, ql, off))
    out = buffer_like(np.full(total * row + 8, 7.0, np.float32))
    capi.check(capi.lib().kvflux_paged_prefill_batch(kc.ptr, vc.ptr, blocks, kv_heads, bs, D, code, td.ptr, width,
                                                     kd.ptr, ld.ptr, sd.ptr, len(seqs), int(ql.max()), int(kv.max()),
                                                     q_heads, qd.ptr, out.ptr, None))
    device.synchronize()
    got = out.download(np.float32)
    assert np.all(got[total * row:] == 7.0)
    got = got[:total * row]
    rows = np.concatenate([np.full(b, i) for i, (_, b) in enumerate(seqs)])
    lens = np.concatenate([np.arange(a - b + 1, a + 1) for a, b in seqs]).astype(np.uint64)
    exp = oracle.paged_attention_rows(kc.download(host), vc.download(host), kv_heads, bs, D, code,
                                      table[rows].reshape(-1), width, lens, q, q_heads, threads=8)
    assert np.all(np.isfinite(got))
    assert np.abs(got - exp).max() < (1e-5 if name == "Float32" else 2e-2)


SINGLE = [  # name, kv heads, q heads, D, block size, kv tokens, query tokens
    ("BFloat16", 2, 8, 128, 16, 33, 33),
    ("BFloat16", 2, 8, 128, 16, 1500, 20),     # key splits beside the parts
    ("Float16", 4, 28, 128, 16, 257, 257),
    ("Float16", 1, 2, 64, 32, 1000, 16),
    ("Float32", 4, 16, 128, 16, 2000, 128),
    ("BFloat16", 1, 4, 64, 8, 640, 640),
]


@pytest.mark.parametrize("case", range(len(SINGLE)))
def test_exact_key_parts(gpu, case):
    name, kv_heads, q_heads, D, bs, kv, tq = SINGLE[case]
    code, host = DTYPES[name]
    kc, vc, blocks, table, width = arena(name, kv_heads, bs, D, [kv], 800 + 2 * case)
    q = oracle.random_elements(0, tq * q_heads * D, oracle.F32, 1, 850 + case)
    need = C.c_size_t(0)
    capi.check(capi.lib().kvflux_paged_prefill_workspace_size(kv_heads, D, kv, tq, q_heads, C.byref(need)))
    exp = oracle.paged_attention_causal(kc.download(host), vc.download(host), kv_heads, bs, D, code, table[0], kv, q,
                                        tq, q_heads, threads=8)
    td, qd = buffer_like(table.reshape(-1)), buffer_like(q)
    for size in (need.value, 0):  # with and without room for key splits
        ws = buffer_like(np.full(size // 4 + 8, np.nan, np.float32))
        out = buffer_like(np.full(q.size + 8, 7.0, np.float32))
        capi.check(capi.lib().kvflux_paged_prefill_exact(kc.ptr, vc.ptr, blocks, kv_heads, bs, D, code, td.ptr, width,
                                                         kv, tq, q_heads, qd.ptr, out.ptr, ws.ptr if size else None,
                                                         size, None))
        device.synchronize()
        got = out.download(np.float32)
        assert np.all(got[q.size:] == 7.0) and np.all(np.isnan(ws.download(np.float32)[size // 4:]))
        assert np.abs(got[:q.size] - exp).max() < 1e-5
